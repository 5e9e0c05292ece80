"""GPU parity of the mask choice of few very wide rows with one threshold, on both sides of
where a wave per row takes them, and of narrow elements, whose masks' bits are not counted."""
import numpy as np
import pytest
import torch

from test_gpu_preprocess_slices import check, rows_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,v,w", [(1, 2049, 8), (341, 2049, 8), (342, 2049, 8), (100, 4097, 8), (80, 20501, 4),
                                   (81, 20501, 4)])
@pytest.mark.parametrize("threshold", [0.9, None])
def test_few_wide_rows(oracle, n, v, w, threshold):
    print("few wide", n, v, w, threshold, flush=True)
    check(oracle, rows_of(n, v, w, n + v), threshold, offset=1)


@pytest.mark.parametrize("n,v,w", [(3, 3000, 2), (70, 65, 1)])
def test_narrow_elements(oracle, n, v, w):
    import invariantbitpacking_amd as ibp
    x = rows_of(n, v, w, v)
    om, ob, _, _ = oracle.preprocess(x, None)
    mask, bitval = ibp.preprocess(torch.from_numpy(x.view("i%d" % w)).cuda(), None)
    assert np.array_equal(mask.cpu().numpy().view(om.dtype), om)
    assert np.array_equal(bitval.cpu().numpy().view(ob.dtype), ob)
