"""GPU parity of the mask choice where rows are scored in slices of 16-byte
chunks: every slice width and number of waves per tile, rows that do not end
with a chunk, tiles that do not end with a row, thresholds that flag nothing."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def rows_of(n, v, w, seed):
    """Columns whose bits are constant in 60 % to all of the rows; some are random."""
    rng = np.random.default_rng(seed)
    base = rng.integers(0, 256, size=(1, v * w), dtype=np.uint8)
    share = rng.choice([0.0, 0.02, 0.08, 0.2, 0.4, 1.0], size=(1, v * w))
    x = np.where(rng.random((n, v * w)) < share, rng.integers(0, 256, size=(n, v * w), dtype=np.uint8), base)
    return np.ascontiguousarray(x).view("u%d" % w)


def check(oracle, x, threshold, offset=0):
    from invariantbitpacking_amd import _capi
    n, v = x.shape
    w = x.dtype.itemsize
    thr = -1.0 if threshold is None else threshold
    room = torch.zeros(n * v + offset, dtype={4: torch.int32, 8: torch.int64}[w], device="cuda")
    t = room[offset:].view(n, v)
    t.copy_(torch.from_numpy(x.view("i%d" % w)))
    mask, bitval = torch.zeros(v, dtype=t.dtype, device="cuda"), torch.zeros(v, dtype=t.dtype, device="cuda")
    step = torch.full((1,), -7, dtype=torch.int32, device="cuda")
    size = _capi.lib().ibp_preprocess_workspace_size(w, v, thr)
    ws = torch.full((size,), 0xa5, dtype=torch.uint8, device="cuda")
    _capi.call("ibp_preprocess", w, t.data_ptr(), n, v, thr, mask.data_ptr(), bitval.data_ptr(), step.data_ptr(),
               ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream)
    om, ob, ostep, _ = oracle.preprocess(x, threshold)
    assert int(step[0]) == ostep
    assert np.array_equal(mask.cpu().numpy().view(om.dtype), om)
    assert np.array_equal(bitval.cpu().numpy().view(ob.dtype), ob)


# (rows, columns) of 4-byte words: 1 to 5, 6 to 8, ... chunks of 16 bytes, whole and not
SHAPES = [(1, 4), (63, 5), (64, 3), (65, 20), (300, 21), (70, 32), (129, 33), (64, 40), (200, 41), (130, 56), (65, 57),
          (500, 64), (300, 65), (64, 80), (200, 81), (130, 100), (129, 112), (257, 113), (300, 130), (64, 256), (65, 257),
          (100, 289), (3, 1027), (1000, 527), (33000, 261)]


@pytest.mark.parametrize("threshold", [None, 0.9, 0.3])
@pytest.mark.parametrize("shape", SHAPES)
def test_mask_choice(oracle, shape, threshold):
    n, v = shape
    print("preprocess slices", shape, threshold, flush=True)
    check(oracle, rows_of(n, v, 4, n + v), threshold, offset=1)
    if v > 3:
        check(oracle, rows_of(n, (v + 1) // 2, 8, n * v), threshold, offset=1)


@pytest.mark.parametrize("n,v,w", [(2000000, 4, 4), (700001, 50, 4), (400003, 25, 8), (20000, 4096, 4)])
def test_mask_choice_of_many_rows(oracle, n, v, w):
    """More tiles than waves in flight."""
    print("preprocess slices", n, v, w, flush=True)
    check(oracle, rows_of(n, v, w, v), None)


def test_nothing_to_save(oracle):
    rng = np.random.default_rng(3)
    check(oracle, rng.integers(0, 1 << 32, size=(5000, 37), dtype=np.uint32), None)
