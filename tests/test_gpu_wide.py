"""GPU parity of the fetch of rows of more than 64 elements of 4 and 8 bytes at
the edges of its chunks (512 bytes), spans (64 chunks) and batches (8 rows):
partial chunks, batches of every size, masks of few and of many runs, packed,
raw and out-of-range rows in one batch, mask rows that change inside a batch."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ibp():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import invariantbitpacking_amd as m
    return m


def masks_of(kind, v, w, rng):
    """Mask words: at most two runs of masked bits per 32 bits, or scattered bits."""
    bits = 8 * w
    m = np.zeros(v, dtype="u%d" % w)
    for j in range(v):
        if kind == "runs" or (kind == "mixed" and j % 7):
            for half in range(bits // 32):
                a, b = sorted(rng.integers(0, 33, size=2))
                m[j] |= np.array(((1 << int(b)) - (1 << int(a))) << (32 * half), dtype=np.uint64).astype(m.dtype)
        else:
            m[j] = (int(rng.integers(0, 2 ** 63)) * 3) % (1 << bits)
    m[0] = ~m.dtype.type(0)  # a column with no free bit
    if v > 1:
        m[v - 1] = 0         # and one with no masked bit
    return m


def rows_for(n, mask, bitval, rng, hit=0.9):
    """Rows whose elements match the masked bits with probability `hit`; every fifth row is random (raw)."""
    x = rng.integers(0, 2 ** 63, size=(n, mask.size), dtype=np.uint64).astype(mask.dtype) * mask.dtype.type(5)
    match = (x & ~mask) | bitval
    take = rng.random(x.shape) < hit
    take[4::5] = False
    return np.where(take, match, x)


# 4-byte elements: 128 a chunk, 8192 a span; 8-byte ones: 64 and 4096
@pytest.mark.parametrize("w,v", [(4, 65), (4, 127), (4, 128), (4, 129), (4, 1025), (4, 8192), (4, 8333),
                                 (8, 65), (8, 127), (8, 128), (8, 513), (8, 4096), (8, 4161)])
@pytest.mark.parametrize("kind", ["runs", "mixed"])
def test_wide_rows_match(ibp, oracle, w, v, kind):
    rng = np.random.default_rng(1000 * w + v)
    n = 43
    dt = np.dtype("i%d" % w)
    mask = masks_of(kind, v, w, rng)
    bitval = rng.integers(0, 2 ** 63, size=v, dtype=np.uint64).astype(mask.dtype) & mask
    x = rows_for(n, mask, bitval, rng).view(dt)
    comp, bm = oracle.compress(x, mask.view(dt), bitval.view(dt))
    stream, off = oracle.compress_condensed(x, mask.view(dt), bitval.view(dt))
    args = [torch.from_numpy(mask.view(dt)).cuda(), torch.from_numpy(bitval.view(dt)).cuda()]
    bmd = torch.from_numpy(bm.view(np.int32)).cuda()
    dev = torch.device("cuda")
    for where in ("device", "pinned"):
        to = (lambda t: t.cuda()) if where == "device" else (lambda t: t.pin_memory())
        cd = to(torch.from_numpy(comp.view(dt)))
        sd, od = to(torch.from_numpy(stream.view(dt))), to(torch.from_numpy(off))
        for picks in (1, 2, 7, 8, 9, n):
            idx = rng.integers(0, n, size=picks)
            want = x[idx]
            for it in (torch.int64, torch.int32):
                ix = torch.from_numpy(idx).to(it).cuda()
                got = ibp.decompress_fetch(cd, *args, bmd, dev, None, ix)
                assert torch.equal(got.cpu(), torch.from_numpy(want)), (where, picks, it)
                got = ibp.decompress(sd, od, *args, dev, v, ix)
                assert torch.equal(got.cpu(), torch.from_numpy(want)), (where, picks, it)
        ibp.index_errors(reset=True)
        idx = np.array([3, n, 4, -1, 0, 9, 14, 1, 2, 5])
        got = ibp.decompress_fetch(cd, *args, bmd, dev, None, torch.from_numpy(idx).cuda()).cpu().numpy()
        assert ibp.index_errors(reset=True) == 2
        ok = (idx >= 0) & (idx < n)
        assert np.array_equal(got[ok], x[idx[ok]]) and not got[~ok].any()
    # the same rows through a plan (one wave per batch of rows)
    out = torch.empty((n, v), dtype=args[0].dtype, device="cuda")
    plan = ibp.BatchedFetch([dict(comp=cd, mask=args[0], bitval=args[1], bitmask=bmd, out=out)])
    plan.launch()
    assert torch.equal(out.cpu(), torch.from_numpy(x))


@pytest.mark.parametrize("w,v", [(4, 200), (8, 65), (8, 4161)])
@pytest.mark.parametrize("k", [2, 5])
def test_wide_clusters_inside_a_batch(ibp, oracle, w, v, k):
    rng = np.random.default_rng(w + v + k)
    n = 41
    dt = np.dtype("i%d" % w)
    mask = np.stack([masks_of("runs" if c else "mixed", v, w, rng) for c in range(k)])
    bitval = rng.integers(0, 2 ** 63, size=(k, v), dtype=np.uint64).astype(mask.dtype) & mask
    cl = np.sort(rng.integers(0, k, size=n)).astype(np.int32)
    cl[::6] = rng.integers(0, k, size=cl[::6].size)  # stretches of one row and of many
    x = np.concatenate([rows_for(n, mask[c], bitval[c], rng)[i:i + 1] for i, c in enumerate(cl)]).view(dt)
    comp, bm = oracle.compress(x, mask.view(dt), bitval.view(dt), clusters=cl)
    idx = rng.integers(0, n, size=29)
    for ix in (None, idx):
        got = ibp.decompress_fetch(torch.from_numpy(comp.view(dt)).cuda(), torch.from_numpy(mask.view(dt)).cuda(),
                                   torch.from_numpy(bitval.view(dt)).cuda(), torch.from_numpy(bm.view(np.int32)).cuda(),
                                   torch.device("cuda"), None, None if ix is None else torch.from_numpy(ix).cuda(),
                                   clusters=torch.from_numpy(cl).cuda())
        assert torch.equal(got.cpu(), torch.from_numpy(x if ix is None else x[ix]))


# team sizes (1, 2, 4, 8 waves) follow from the chunks and the rows; 32 KiB is the widest row a team packs
# (here rows of 512 columns to 32 KiB go to teams, of eight waves; test_gpu_pack_teams.py has the other teams)
@pytest.mark.parametrize("w,v", [(4, 65), (4, 129), (4, 255), (4, 513), (4, 2049), (4, 8192), (4, 8193),
                                 (8, 65), (8, 127), (8, 256), (8, 257), (8, 1030), (8, 4096), (8, 4097)])
@pytest.mark.parametrize("n", [37, 4500])
def test_wide_pack_matches_oracle(ibp, oracle, w, v, n):
    if n > 1000 and v > 300:
        n = 70  # many rows only where they change the team
    rng = np.random.default_rng(77 * w + v + n)
    dt = np.dtype("i%d" % w)
    k = 3
    mask = np.stack([masks_of(kind, v, w, rng) for kind in ("runs", "mixed", "runs")])
    bitval = rng.integers(0, 2 ** 63, size=(k, v), dtype=np.uint64).astype(mask.dtype) & mask
    cl = rng.integers(0, k, size=n).astype(np.int32)
    by = [rows_for(n, mask[c], bitval[c], rng) for c in range(k)]
    x = np.stack(by)[cl, np.arange(n)].view(dt)
    m, b = mask.view(dt), bitval.view(dt)
    md, bd, cd = torch.from_numpy(m).cuda(), torch.from_numpy(b).cuda(), torch.from_numpy(cl).cuda()
    for clusters in (cl, None):
        kw = {} if clusters is None else {"clusters": cd}
        mm, bb = (m, b) if clusters is not None else (m[1], b[1])
        mmd, bbd = (md, bd) if clusters is not None else (md[1].contiguous(), bd[1].contiguous())
        comp, bm = oracle.compress(x, mm, bb, clusters=clusters)
        t = torch.from_numpy(x).cuda()
        got = ibp.compress_inplace(t, mmd, bbd, **kw)
        assert np.array_equal(got.cpu().numpy(), bm.view(np.int32))
        assert np.array_equal(t.cpu().numpy().view(comp.dtype), comp)
        stream, off = oracle.compress_condensed(x, mm, bb, clusters=clusters)
        s, o = ibp.compress_condensed(torch.from_numpy(x).cuda(), mmd, bbd, **kw)
        assert np.array_equal(o.cpu().numpy(), off) and np.array_equal(s.cpu().numpy().view(stream.dtype), stream)
    idx = rng.integers(0, n, size=n // 2)
    want, wbm = oracle.compress(x[idx], m[1], b[1])
    t = torch.from_numpy(x).cuda()
    got = ibp.compress_inplace(t, md[1].contiguous(), bd[1].contiguous(), torch.from_numpy(idx).cuda())
    assert np.array_equal(got.cpu().numpy(), wbm.view(np.int32))
    assert np.array_equal(t.cpu().numpy()[:n // 2].view(want.dtype), want)
