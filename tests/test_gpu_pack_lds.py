"""Pack of few rows whose slot buffers fill a CU's LDS to the last byte: rows of
a whole fraction of 160 KiB, where the buffers of as many waves as fit and the
kernel's own variable have to share it."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,v", [(1, 16384), (2, 8192), (1, 20480), (2, 10240), (1, 40960), (4, 10240), (8, 5120)])
def test_rows_of_a_fraction_of_lds(oracle, w, v):
    import invariantbitpacking_amd as ibp
    rng = np.random.default_rng(v + w)
    dt = np.dtype("i%d" % w)
    x = rng.integers(0, 256, size=(37, v * w), dtype=np.uint8)
    x[:, ::2] &= 3
    mask = np.zeros(v * w, np.uint8)
    mask[::2] = 0xfc
    x, mask = x.view(dt), mask.view(dt)
    comp, bm = oracle.compress(x, mask, np.zeros_like(mask))
    t = torch.from_numpy(x.copy()).cuda()
    print("pack lds", w, v, flush=True)
    got = ibp.compress_inplace(t, torch.from_numpy(mask).cuda(), torch.zeros(v, dtype=t.dtype, device="cuda"))
    assert np.array_equal(got.cpu().numpy().view(np.uint32), bm.view(np.uint32))
    assert np.array_equal(t.cpu().numpy().view(comp.dtype), comp)
