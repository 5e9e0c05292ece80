"""GPU parity of the fetch and pack by teams of waves where they are chosen by
size: many rows of 65 to 511 columns, and windows of rows of several mask rows (batches of
one mask row, raw rows, single rows, refused rows), in every window size."""
import numpy as np
import pytest
import torch

from test_gpu_wide import masks_of, rows_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ibp():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import invariantbitpacking_amd as m
    return m


def expect(x, idx, good=None):
    ok = (idx >= 0) & (idx < len(x))
    if good is not None:
        ok &= good[np.clip(idx, 0, len(x) - 1)]
    want = x[np.clip(idx, 0, len(x) - 1)].copy()
    want[~ok] = 0
    return want


def fetch_all(ibp, oracle, x, mask, bitval, idx, clusters=None, bad=None):
    """Slots and stream of x by index, against the rows themselves."""
    kw = {} if clusters is None else {"clusters": clusters}
    comp, bm = oracle.compress(x, mask, bitval, **kw)
    stream, off = oracle.compress_condensed(x, mask, bitval, **kw)
    good = None
    if clusters is not None:
        cl = clusters.copy()
        if bad is not None:
            cl[bad] = [-1, mask.shape[0], 1 << 30][: len(bad)]
            good = (cl >= 0) & (cl < mask.shape[0])
        kw = {"clusters": torch.from_numpy(cl).cuda()}
    want = expect(x, idx, good)
    m, b = torch.from_numpy(mask).cuda(), torch.from_numpy(bitval).cuda()
    i = torch.from_numpy(idx).cuda()
    dev = torch.device("cuda")
    got = ibp.decompress_fetch(torch.from_numpy(comp).cuda(), m, b, torch.from_numpy(bm.view(np.int32)).cuda(), dev,
                               x.shape[1], i, **kw)
    assert np.array_equal(got.cpu().numpy(), want), "slots"
    got = ibp.decompress(torch.from_numpy(stream).cuda(), torch.from_numpy(off).cuda(), m, b, dev, x.shape[1], i, **kw)
    assert np.array_equal(got.cpu().numpy().reshape(want.shape), want), "stream"


@pytest.mark.parametrize("w,v", [(4, 65), (4, 127), (4, 128), (4, 129), (4, 300), (8, 65), (8, 128), (8, 129), (8, 511)])
def test_many_rows(ibp, oracle, w, v):
    rng = np.random.default_rng(100 * w + v)
    dt = np.dtype("i%d" % w)
    mask = masks_of("mixed" if v % 2 else "runs", v, w, rng)
    bitval = rng.integers(0, 2 ** 63, size=v, dtype=np.uint64).astype(mask.dtype) & mask
    x = rows_for(301, mask, bitval, rng).view(dt)
    n = (8 << 20) // (v * w) + 5
    idx = rng.integers(0, 301, size=n)
    idx[[0, 7, n - 1]] = [-1, 301, 1 << 40]
    print("teams", w, v, n, flush=True)
    fetch_all(ibp, oracle, x, mask.view(dt), bitval.view(dt), idx)
    fetch_all(ibp, oracle, x, mask.view(dt), bitval.view(dt), rng.integers(0, 301, size=n - 200).astype(np.int32))


@pytest.mark.parametrize("w,v", [(4, 1536), (4, 1537), (8, 768), (8, 1025)])
@pytest.mark.parametrize("k,n", [(1, 3), (2, 600), (16, 700), (3, 1500), (16, 2500), (16, 5000), (2, 9000), (5, 9001),
                                 (16, 40001)])
def test_windows_of_mask_rows(ibp, oracle, w, v, k, n):
    rng = np.random.default_rng(w + v + 10 * n + k)
    dt = np.dtype("i%d" % w)
    mask = np.stack([masks_of("mixed" if c % 3 else "runs", v, w, rng) for c in range(k)])
    bitval = rng.integers(0, 2 ** 63, size=mask.shape, dtype=np.uint64).astype(mask.dtype) & mask
    cl = rng.integers(0, k, size=203).astype(np.int32)
    x = np.zeros((203, v), mask.dtype)
    for c in range(k):
        x[cl == c] = rows_for(int((cl == c).sum()), mask[c], bitval[c], rng)
    idx = rng.integers(0, 203, size=n)
    idx[n // 2] = 203
    bad = rng.choice(203, size=3, replace=False) if k > 1 else None
    print("windows", w, v, k, n, flush=True)
    fetch_all(ibp, oracle, x.view(dt), mask.view(dt), bitval.view(dt), idx, cl, bad)


@pytest.mark.parametrize("w,v", [(4, 65), (4, 129), (8, 65), (8, 128)])
def test_pack_of_many_rows(ibp, oracle, w, v):
    rng = np.random.default_rng(10 * w + v)
    dt = np.dtype("i%d" % w)
    mask = np.stack([masks_of("mixed", v, w, rng) for _ in range(2)])
    bitval = rng.integers(0, 2 ** 63, size=mask.shape, dtype=np.uint64).astype(mask.dtype) & mask
    n = 32768 + 33
    cl = (rng.random(n) < 0.3).astype(np.int32)
    x = np.where(cl[:, None] == 0, rows_for(n, mask[0], bitval[0], rng), rows_for(n, mask[1], bitval[1], rng)).view(dt)
    m, b = mask.view(dt), bitval.view(dt)
    print("pack teams", w, v, flush=True)
    for mm, bb, kw, kd in ((m[0].copy(), b[0].copy(), {}, {}),
                           (m, b, {"clusters": cl}, {"clusters": torch.from_numpy(cl).cuda()})):
        comp, bm = oracle.compress(x, mm, bb, **kw)
        t = torch.from_numpy(x.copy()).cuda()
        got = ibp.compress_inplace(t, torch.from_numpy(mm).cuda(), torch.from_numpy(bb).cuda(), **kd)
        assert np.array_equal(got.cpu().numpy().view(np.uint32), bm.view(np.uint32))
        assert np.array_equal(t.cpu().numpy().view(comp.dtype), comp)
