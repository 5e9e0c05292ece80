"""GPU parity of the compressed sizes of whole tables (rows in slices of
16-byte chunks: every slice width and number of waves per tile, rows that do
not end with a chunk) and of their running sums at the edges of its tiles."""
import numpy as np
import pytest
import torch

from test_gpu_preprocess_slices import SHAPES, rows_of

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ibp():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import invariantbitpacking_amd as m
    return m


def masks_of(x, seed):
    """Masks of the bits that 9 of 10 rows share, some columns without any."""
    rng = np.random.default_rng(seed)
    w = x.dtype.itemsize
    bits = np.unpackbits(x[:2000].view(np.uint8), axis=1).mean(axis=0)
    m = np.packbits(((bits > 0.9) | (bits < 0.1)).astype(np.uint8)).view("u%d" % w)
    b = np.packbits((bits > 0.9).astype(np.uint8)).view("u%d" % w)
    off = rng.random(m.shape[0]) < 0.2
    m[off] = 0
    b[off] = 0
    return m, b


@pytest.mark.parametrize("shape", SHAPES)
def test_sizes_of_a_table(ibp, oracle, shape):
    n, v = shape
    print("sizes", shape, flush=True)
    for x in [rows_of(n, v, 4, n + v)] + ([rows_of(n, (v + 1) // 2, 8, n * v)] if v > 3 else []):
        w = x.dtype.itemsize
        m, b = masks_of(x, v)
        want, _ = oracle.get_compress_size(x, m, b)
        room = torch.zeros(x.size + 1, dtype={4: torch.int32, 8: torch.int64}[w], device="cuda")
        t = room[1:].view(x.shape)
        t.copy_(torch.from_numpy(x.view("i%d" % w)))
        total = torch.full((1,), 5, dtype=torch.int64, device="cuda")
        got = ibp.get_compress_size(t, torch.from_numpy(m.view("i%d" % w)).cuda(),
                                    torch.from_numpy(b.view("i%d" % w)).cuda(), None, total)
        assert np.array_equal(got.cpu().numpy(), want)
        assert int(total[0]) == 5 + int(want.sum())


@pytest.mark.parametrize("n", [1, 255, 4095, 4096, 4097, 65537, 8388608 + 1, 8388608 + 8192])
def test_running_sums(ibp, n):
    """Offsets are the running sums of the sizes; above 2048 tiles of 4096 rows these are scanned first."""
    print("running sums", n, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randint(0, 1 << 30, (n, 4), generator=g, device="cuda", dtype=torch.int32)
    x[torch.rand((n,), generator=g, device="cuda") < 0.7] &= 0xff
    mask = torch.full((4,), 0x3fffff00, dtype=torch.int32, device="cuda")
    bitval = torch.zeros(4, dtype=torch.int32, device="cuda")
    sizes = ibp.get_compress_size(x, mask, bitval)
    assert n < 300 or sizes.unique().numel() > 1
    _, offsets = ibp.compress_condensed(x, mask, bitval)
    assert torch.equal(offsets.to("cuda"), torch.cumsum(sizes.to("cuda"), 0))
