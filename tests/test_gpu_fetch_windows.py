"""GPU parity of the clustered fetch by teams of waves in each way it takes its rows: one row
a batch, whole windows (all rows alike, or two waves a row), parts of windows with the rest by
a wave per row; rows of one and of two spans of chunks, raw and refused rows, pinned rows."""
import numpy as np
import pytest
import torch

from test_gpu_fetch_teams import expect
from test_gpu_wide import masks_of, rows_for

pytestmark = pytest.mark.gpu

ROWS = 131  # of the table


@pytest.fixture(scope="module")
def ibp():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import invariantbitpacking_amd as m
    return m


def table(w, v, k, usage, rng):
    mask = np.stack([masks_of("mixed" if c % 3 else "runs", v, w, rng) for c in range(k)])
    bitval = rng.integers(0, 2 ** 63, size=mask.shape, dtype=np.uint64).astype(mask.dtype) & mask
    cl = rng.integers(0, k, size=ROWS).astype(np.int32)
    if usage == "one":
        cl[:] = k - 1
    elif usage == "mostly":
        cl[rng.random(ROWS) < 0.9] = 0
    x = np.zeros((ROWS, v), mask.dtype)
    for c in range(k):
        if (cl == c).any():
            x[cl == c] = rows_for(int((cl == c).sum()), mask[c], bitval[c], rng)
    raw = rng.random(ROWS) < 0.15
    x[raw] = rng.integers(0, 2 ** 63, size=(int(raw.sum()), v), dtype=np.uint64).astype(mask.dtype)
    return x, mask, bitval, cl


@pytest.mark.parametrize("usage", ["one", "mostly", "even"])
# 32 KiB and more: two spans of 64 chunks
@pytest.mark.parametrize("w,v", [(4, 1537), (8, 800), (4, 8200), (8, 4133)])
# one row a batch (teams of eight, four); windows of four, eight; parts of windows of 16 (with
# a last window of 1, of 7 rows)
@pytest.mark.parametrize("n", [1, 512, 1000, 1025, 2049, 4096, 4097, 4103])
def test_rows_by_cluster_use(ibp, oracle, usage, w, v, n):
    rng = np.random.default_rng(w * v + n + len(usage))
    x, mask, bitval, cl = table(w, v, 5, usage, rng)
    dt = np.dtype("i%d" % w)
    comp, bm = oracle.compress(x.view(dt), mask.view(dt), bitval.view(dt), clusters=cl)
    stream, off = oracle.compress_condensed(x.view(dt), mask.view(dt), bitval.view(dt), clusters=cl)
    bad = cl.copy()
    bad[rng.choice(ROWS, size=2, replace=False)] = [-1, 5]
    idx = rng.integers(0, ROWS, size=n)
    if n > 1:
        idx[rng.choice(n, size=2, replace=False)] = [-1, ROWS]
    want = expect(x.view(dt), idx, (bad >= 0) & (bad < 5))
    dev = torch.device("cuda")
    m, b, c = (torch.from_numpy(a).cuda() for a in (mask.view(dt), bitval.view(dt), bad))
    bits = torch.from_numpy(bm.view(np.int32)).cuda()
    print("cluster use", usage, w, v, n, flush=True)
    ibp.index_errors(reset=True)
    wrong = int((~((idx >= 0) & (idx < ROWS))).sum() + ((idx >= 0) & (idx < ROWS) & ((bad < 0) | (bad > 4))[idx % ROWS]).sum())
    for ix in (torch.from_numpy(idx).cuda(), torch.from_numpy(idx.astype(np.int32)).cuda()):
        for rows in (torch.from_numpy(comp).cuda(), torch.from_numpy(comp).pin_memory()):
            got = ibp.decompress_fetch(rows, m, b, bits, dev, v, ix, clusters=c)
            assert np.array_equal(got.cpu().numpy(), want), "slots"
            assert ibp.index_errors(reset=True) == wrong
        got = ibp.decompress(torch.from_numpy(stream).cuda(), torch.from_numpy(off).cuda(), m, b, dev, v, ix, clusters=c)
        assert np.array_equal(got.cpu().numpy().reshape(want.shape), want), "stream"
        assert ibp.index_errors(reset=True) == wrong


# windows of 16, 32 and 64 rows; whether they go to teams is read from four stretches of 16 rows
@pytest.mark.parametrize("n", [4200, 9001, 20003])
@pytest.mark.parametrize("order", ["sampled alike", "sampled mixed", "sorted", "refused"])
def test_rows_unlike_the_sample(ibp, oracle, n, order):
    rng = np.random.default_rng(n + len(order))
    x, mask, bitval, cl = table(8, 800, 5, "even", rng)
    comp, bm = oracle.compress(x.view("i8"), mask.view("i8"), bitval.view("i8"), clusters=cl)
    idx = rng.integers(0, ROWS, size=n)
    packed = np.unpackbits(bm.view(np.uint8), bitorder="little")[:ROWS] == 1
    of = [np.flatnonzero((cl == c) & packed) for c in range(5)]
    sample = (np.arange(64) // 16 * (n // 4) + np.arange(64) % 16)
    if order == "sampled alike":
        idx[sample] = rng.choice(of[0], size=64)
    elif order == "sampled mixed":
        idx = rng.choice(of[1], size=n)
        idx[sample] = rng.integers(0, ROWS, size=64)
    elif order == "sorted":
        idx = idx[np.argsort(cl[idx], kind="stable")]
    else:
        idx[sample] = -1
    args = [torch.from_numpy(a).cuda() for a in (comp.view("i8"), mask.view("i8"), bitval.view("i8"), bm.view(np.int32))]
    print("unlike the sample", n, order, flush=True)
    got = ibp.decompress_fetch(*args, torch.device("cuda"), None, torch.from_numpy(idx).cuda(),
                               clusters=torch.from_numpy(cl).cuda())
    assert np.array_equal(got.cpu().numpy(), expect(x.view("i8"), idx))
