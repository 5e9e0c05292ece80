"""GPU parity of the fetch of narrow wide rows from pinned host memory, on both sides of where
teams of waves read them."""
import re

import numpy as np
import pytest
import torch

from test_gpu_wide import masks_of, rows_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,v,n,team", [(8, 65, 16200, False), (8, 128, 8200, False), (8, 159, 6600, False),
                                        (8, 160, 6600, True), (8, 160, 6500, False), (4, 65, 33000, True),
                                        (4, 159, 13200, True)])
@pytest.mark.parametrize("condensed", [False, True])
def test_pinned_rows(oracle, capfd, w, v, n, team, condensed):
    import invariantbitpacking_amd as ibp
    rng = np.random.default_rng(v + n)
    dt = np.dtype("i%d" % w)
    mask = masks_of("mixed", v, w, rng)
    bitval = rng.integers(0, 2 ** 63, size=v, dtype=np.uint64).astype(mask.dtype) & mask
    x = rows_for(211, mask, bitval, rng).view(dt)
    m, b = mask.view(dt), bitval.view(dt)
    idx = rng.integers(0, 211, size=n)
    idx[[0, n - 1]] = [211, -1]
    want = x[np.clip(idx, 0, 210)]
    want[[0, n - 1]] = 0
    gpu = torch.device("cuda")
    tm, tb, ti = (torch.from_numpy(a.copy()).to(gpu) for a in (m, b, idx))
    print("pinned fetch", w, v, n, condensed, flush=True)
    if condensed:
        data, offsets = oracle.compress_condensed(x, m, b)
        call = lambda c: ibp.decompress(c, torch.from_numpy(offsets).to(gpu), tm, tb, gpu, v, ti)
    else:
        data, bits = oracle.compress(x, m, b)
        call = lambda c: ibp.decompress_fetch(c, tm, tb, torch.from_numpy(bits.view(np.int32)).to(gpu), gpu, v, ti)
    comp = torch.from_numpy(data).pin_memory()
    ibp.print_debug(True)
    try:
        capfd.readouterr()
        got = call(comp)
        torch.cuda.synchronize()
        out = capfd.readouterr().out
    finally:
        ibp.print_debug(False)
    kind, place = re.search(r"decompress_fetch: ([a-z ]+), impl [-0-9]+, ([a-z]+) ", out).groups()
    assert (kind, place) == ("team of waves per batch of rows" if team else "wave per row", "host"), out
    assert np.array_equal(got.cpu().numpy().reshape(want.shape), want)
