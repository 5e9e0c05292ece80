"""Calls that pick their kernels by size or place, captured in a graph: every replay, on new
contents of the captured buffers, equals the eager call."""
import numpy as np
import pytest
import torch

from test_gpu_fetch_windows import ROWS, table
from test_gpu_preprocess_slices import rows_of

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ibp():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import invariantbitpacking_amd as m
    return m


def replays(capture, refill, check, times=3):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        capture()  # outside the graph first
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        capture()
    for k in range(times):
        refill(k)
        g.replay()
        torch.cuda.synchronize()
        check(k)


@pytest.mark.parametrize("n", [600, 3000, 9000])
def test_fetch_by_cluster_use(ibp, oracle, n):
    rng = np.random.default_rng(n)
    v, dt = 800, np.dtype("i8")
    x, mask, bitval, cl = table(8, v, 5, "mostly", rng)
    comp, bm = oracle.compress(x.view(dt), mask.view(dt), bitval.view(dt), clusters=cl)
    c, m, b, bits, cld = (torch.from_numpy(a).cuda() for a in (comp.view(dt), mask.view(dt), bitval.view(dt),
                                                               bm.view(np.int32), cl))
    rows = torch.from_numpy(x.view(dt)).cuda()
    idx = torch.zeros(n, dtype=torch.int64, device="cuda")
    out = torch.empty((n, v), dtype=torch.int64, device="cuda")
    dev = torch.device("cuda")
    print("captured fetch", n, flush=True)

    def refill(k):
        idx.copy_(torch.from_numpy(rng.integers(0, ROWS, size=n)))
        out.fill_(-1)

    def check(k):
        assert torch.equal(out, rows[idx])

    replays(lambda: ibp.decompress_fetch(c, m, b, bits, dev, v, idx, None, None, None, out, clusters=cld), refill, check)


@pytest.mark.parametrize("n,v", [(700, 700), (5000, 700), (33000, 100)])
def test_pack(ibp, oracle, n, v):
    from invariantbitpacking_amd import _capi
    xs = [rows_of(n, v, 8, k) for k in range(3)]
    om, ob, _, _ = oracle.preprocess(xs[0], 0.9)
    want = [oracle.compress(x, om, ob) for x in xs]
    m, b = torch.from_numpy(om.view("i8")).cuda(), torch.from_numpy(ob.view("i8")).cuda()
    t = torch.zeros((n, v), dtype=torch.int64, device="cuda")
    bits = torch.zeros((n + 31) // 32, dtype=torch.int32, device="cuda")
    print("captured pack", n, v, flush=True)

    def refill(k):
        t.copy_(torch.from_numpy(xs[k].view("i8")))
        bits.fill_(-1)

    def check(k):
        assert np.array_equal(bits.cpu().numpy().view(np.uint32), want[k][1].view(np.uint32))
        assert np.array_equal(t.cpu().numpy().view(want[k][0].dtype), want[k][0])

    replays(lambda: _capi.call("ibp_compress", 8, t.data_ptr(), t.data_ptr(), n, v, m.data_ptr(), b.data_ptr(), None, 8, n,
                               bits.data_ptr(), torch.cuda.current_stream().cuda_stream), refill, check)


@pytest.mark.parametrize("n,v", [(3000, 50), (100, 4097)])
@pytest.mark.parametrize("threshold", [None, 0.9])
def test_preprocess_and_offsets(ibp, oracle, n, v, threshold):
    from invariantbitpacking_amd import _capi
    xs = [rows_of(n, v, 8, 10 + k) for k in range(3)]
    thr = -1.0 if threshold is None else threshold
    t = torch.zeros((n, v), dtype=torch.int64, device="cuda")
    m, b = torch.zeros(v, dtype=torch.int64, device="cuda"), torch.zeros(v, dtype=torch.int64, device="cuda")
    size = _capi.lib().ibp_preprocess_workspace_size(8, v, thr)
    ws = torch.zeros(size, dtype=torch.uint8, device="cuda")
    off = torch.zeros(n, dtype=torch.int64, device="cuda")
    print("captured preprocess", n, v, threshold, flush=True)

    def capture():
        s = torch.cuda.current_stream().cuda_stream
        _capi.call("ibp_preprocess", 8, t.data_ptr(), n, v, thr, m.data_ptr(), b.data_ptr(), None, ws.data_ptr(), size, s)
        _capi.call("ibp_condensed_offsets_noalloc", 8, t.data_ptr(), n, v, m.data_ptr(), b.data_ptr(), None, 8, n,
                   off.data_ptr(), None, s)

    def refill(k):
        t.copy_(torch.from_numpy(xs[k].view("i8")))
        m.zero_()
        b.zero_()

    def check(k):
        om, ob, _, _ = oracle.preprocess(xs[k], threshold)
        assert np.array_equal(m.cpu().numpy().view(om.dtype), om) and np.array_equal(b.cpu().numpy().view(ob.dtype), ob)
        assert np.array_equal(off.cpu().numpy(), oracle.compress_condensed(xs[k], om, ob)[1])

    replays(capture, refill, check)
