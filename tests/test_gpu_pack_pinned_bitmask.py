"""Pack with its bitmask in pinned host memory: the same bits as in device memory, rows that a
wave takes each and rows that go to teams of waves alike."""
import numpy as np
import pytest
import torch

from test_gpu_wide import masks_of, rows_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,v,n", [(8, 64, 70), (8, 600, 70), (4, 1025, 1000), (8, 2752, 33), (4, 65, 32768)])
def test_bitmask_in_pinned_memory(oracle, w, v, n):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from invariantbitpacking_amd import _capi
    rng = np.random.default_rng(v + n)
    dt = np.dtype("i%d" % w)
    mask = masks_of("mixed", v, w, rng)
    bitval = rng.integers(0, 2 ** 63, size=v, dtype=np.uint64).astype(mask.dtype) & mask
    x = rows_for(n, mask, bitval, rng).view(dt)
    comp, bm = oracle.compress(x, mask.view(dt), bitval.view(dt))
    t = torch.from_numpy(x.copy()).cuda()
    m, b = torch.from_numpy(mask.view(dt)).cuda(), torch.from_numpy(bitval.view(dt)).cuda()
    bits = torch.full(((n + 31) // 32,), -1, dtype=torch.int32).pin_memory()
    print("pinned bitmask", w, v, n, flush=True)
    _capi.call("ibp_compress", w, t.data_ptr(), t.data_ptr(), n, v, m.data_ptr(), b.data_ptr(), None, 8, n,
               bits.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert np.array_equal(bits.numpy().view(np.uint32), bm.view(np.uint32))
    assert np.array_equal(t.cpu().numpy().view(comp.dtype), comp)
