"""GPU parity of the pack by teams of waves, in every team size and with several rows per
block: slots in place and by index, condensed streams, a mask row per cluster, raw and refused
rows.  The debug line shows that the team ran."""
import ctypes
import re

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


# teams of 1, 2, 4 and 8 waves (256 CUs); 49200 and more rows of less than 800 bytes; 5000 and
# 4200 rows for 4096 blocks of eight waves, 40000 for 8192 of four
@pytest.mark.parametrize("w,v,n,team", [(8, 65, 49211, 1), (4, 128, 65601, 1), (4, 300, 33001, 2), (4, 512, 3001, 2),
                                        (4, 512, 9001, 2), (8, 300, 40001, 4), (4, 600, 4090, 4), (4, 513, 100, 8),
                                        (8, 600, 5003, 8), (8, 2752, 4201, 8), (4, 8192, 33, 8)])
def test_team(ibp, oracle, capfd, w, v, n, team):
    from invariantbitpacking_amd import _capi
    rng = np.random.default_rng(w + v + n)
    dt = np.dtype("i%d" % w)
    k = 3
    mask = np.stack([masks_of(kind, v, w, rng) for kind in ("runs", "mixed", "runs")])
    bitval = rng.integers(0, 2 ** 63, size=(k, v), dtype=np.uint64).astype(mask.dtype) & mask
    few = 101  # rows that the n repeat; every fifth is raw
    base = np.stack([rows_for(few, mask[c], bitval[c], rng) for c in range(k)])
    cl = rng.integers(0, k, size=n).astype(np.int32)
    x = base[cl, rng.integers(0, few, size=n)].view(dt)
    m, b = np.ascontiguousarray(mask).view(dt), np.ascontiguousarray(bitval).view(dt)
    bad = cl.copy()
    bad[rng.choice(n, size=2, replace=False)] = [-1, k]
    t = torch.from_numpy(x).cuda()
    md, bd, cd, badd = (torch.from_numpy(a).cuda() for a in (m, b, cl, bad))
    stream = torch.cuda.current_stream().cuda_stream

    def pack(out, rows, clusters=None, index=None, offsets=None):
        bits = torch.full(((rows + 31) // 32,), -1, dtype=torch.int32, device="cuda")
        lay = _capi.Layout()
        lay.offsets = None if offsets is None else offsets.data_ptr()
        lay.stream_bytes = 0 if offsets is None else out.numel() * out.element_size()
        lay.clusters = None if clusters is None else clusters.data_ptr()
        lay.num_clusters = 0 if clusters is None else k
        mm, bb = (md, bd) if clusters is not None else (md[1], bd[1])
        src = out if index is None and offsets is None else t
        capfd.readouterr()
        _capi.call("ibp_compress_ex", w, src.data_ptr(), out.data_ptr(), n, v, mm.data_ptr(), bb.data_ptr(),
                   None if index is None else index.data_ptr(), 8 if index is None else index.element_size(), rows,
                   bits.data_ptr(), ctypes.byref(lay), stream)
        torch.cuda.synchronize()
        line = re.search(r"compress: team of ([0-9]+) waves per row, .* n=([0-9]+),", capfd.readouterr().out)
        assert line and int(line.group(1)) == team and int(line.group(2)) == rows
        return bits.cpu().numpy().view(np.uint32)

    print("pack team", w, v, n, team, flush=True)
    ibp.print_debug(True)
    try:
        for clusters, host in ((None, None), (cd, cl)):
            mm, bb = (m, b) if clusters is not None else (m[1].copy(), b[1].copy())
            comp, bm = oracle.compress(x, mm, bb, clusters=host)
            out = t.clone()
            assert np.array_equal(pack(out, n, clusters), bm.view(np.uint32))
            assert np.array_equal(out.cpu().numpy().view(comp.dtype), comp)
            want, off = oracle.compress_condensed(x, mm, bb, clusters=host)
            s = torch.zeros(want.size, dtype=t.dtype, device="cuda")
            assert np.array_equal(pack(s, n, clusters, offsets=torch.from_numpy(off).cuda()), bm.view(np.uint32))
            assert np.array_equal(s.cpu().numpy().view(want.dtype).reshape(want.shape), want)
        # refused rows keep their slots; out of place by index (the same number of rows: the same team)
        comp, bm = oracle.compress(x, m, b, clusters=cl)
        bits = np.unpackbits(bm.view(np.uint8), bitorder="little")[:n]
        idx = rng.integers(0, n, size=n)
        idx[rng.choice(n, size=2, replace=False)] = [-1, n]
        ok = (idx >= 0) & (idx < n)
        ok &= ((bad >= 0) & (bad < k))[idx % n]
        for dtype in (torch.int64, torch.int32):
            out = torch.full((n, v), 77, dtype=t.dtype, device="cuda")
            got = pack(out, n, badd, torch.from_numpy(idx).to(dtype).cuda())
            assert np.array_equal(np.unpackbits(got.view(np.uint8), bitorder="little")[:n], bits[idx % n] & ok)
            rows = out.cpu().numpy()
            assert np.array_equal(rows[ok].view(comp.dtype), comp[idx[ok]]) and (rows[~ok] == 77).all()
    finally:
        ibp.print_debug(False)
