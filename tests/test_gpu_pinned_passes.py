"""GPU parity of the mask choice and the sizes of tables in pinned host memory, which the
kernels read over PCIe, on both sides of where a wave reads each row by itself."""
import numpy as np
import pytest
import torch

from test_gpu_preprocess_slices import rows_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,v,w", [(1001, 39, 8), (1001, 40, 8), (700, 79, 4), (700, 81, 4), (9001, 257, 4), (333, 2752, 8),
                                   (5000, 36, 8), (5000, 37, 8), (5000, 72, 4), (5000, 73, 4)])
def test_pinned_table(oracle, n, v, w):
    from invariantbitpacking_amd import _capi
    x = rows_of(n, v, w, n + v)
    t = torch.from_numpy(x.view("i%d" % w)).pin_memory()
    stream = torch.cuda.current_stream().cuda_stream
    print("pinned", n, v, w, flush=True)
    for threshold in (None, 0.9):
        m, b = torch.zeros(v, dtype=t.dtype, device="cuda"), torch.zeros(v, dtype=t.dtype, device="cuda")
        step = torch.full((1,), -7, dtype=torch.int32, device="cuda")
        _capi.call("ibp_preprocess", w, t.data_ptr(), n, v, -1.0 if threshold is None else threshold, m.data_ptr(),
                   b.data_ptr(), step.data_ptr(), None, 0, stream)
        om, ob, ostep, _ = oracle.preprocess(x, threshold)
        assert int(step[0]) == ostep
        assert np.array_equal(m.cpu().numpy().view(om.dtype), om) and np.array_equal(b.cpu().numpy().view(ob.dtype), ob)
    off = torch.zeros(n, dtype=torch.int64, device="cuda")
    _capi.call("ibp_condensed_offsets", w, t.data_ptr(), n, v, m.data_ptr(), b.data_ptr(), None, 8, n, off.data_ptr(),
               None, stream)
    want = oracle.compress_condensed(x, om, ob)[1]
    assert np.array_equal(off.cpu().numpy(), want)
