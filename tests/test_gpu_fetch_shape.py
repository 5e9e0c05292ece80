"""The launch shape a caller asks for holds for rows that go to teams of waves, and debug mode
reports the shape that is launched."""
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


@pytest.mark.parametrize("w,v,k,n", [(8, 600, 0, 3000), (4, 65, 0, 40000), (8, 800, 3, 700), (8, 800, 3, 3000),
                                     (8, 800, 3, 9000)])
@pytest.mark.parametrize("nblks,nthreads", [(None, None), (None, 64), (None, 128), (None, 192), (3, 256), (7, 1024)])
def test_shape(ibp, oracle, capfd, w, v, k, n, nblks, nthreads):
    rng = np.random.default_rng(v + n)
    dt = np.dtype("i%d" % w)
    mask = np.stack([masks_of("runs", v, w, rng) for _ in range(max(k, 1))])
    bitval = rng.integers(0, 2 ** 63, size=mask.shape, dtype=np.uint64).astype(mask.dtype) & mask
    cl = (np.arange(101) % max(k, 1)).astype(np.int32)
    x = np.zeros((101, v), mask.dtype)
    for c in range(max(k, 1)):
        x[cl == c] = rows_for(int((cl == c).sum()), mask[c], bitval[c], rng)
    m, b = (mask, bitval) if k else (mask[0], bitval[0])
    comp, bm = oracle.compress(x.view(dt), m.view(dt), b.view(dt), **({"clusters": cl} if k else {}))
    idx = rng.integers(0, 101, size=n)
    args = [torch.from_numpy(a).cuda() for a in (comp, m.view(dt).copy(), b.view(dt).copy(), bm.view(np.int32))]
    kw = {"clusters": torch.from_numpy(cl).cuda()} if k else {}
    print("shape", w, v, k, n, nblks, nthreads, flush=True)
    ibp.print_debug(True)
    try:
        capfd.readouterr()
        got = ibp.decompress_fetch(*args, torch.device("cuda"), None, torch.from_numpy(idx).cuda(), nblks, nthreads, **kw)
        torch.cuda.synchronize()
        out = capfd.readouterr().out
    finally:
        ibp.print_debug(False)
    assert np.array_equal(got.cpu().numpy(), x.view(dt)[idx])
    kind, grid, block, rows = re.search(
        r"decompress_fetch: ([a-z ]+), impl.* grid ([0-9]+) x ([0-9]+), rows in flight ([0-9]+)", out).groups()
    grid, block, rows = int(grid), int(block), int(rows)
    assert kind == ("wave per row" if k and nthreads == 64 else "team of waves per batch of rows"), out
    assert block % 64 == 0 and block <= (nthreads or 512)
    if nblks:
        assert grid == nblks
    elif kind.startswith("team"):
        assert rows in (1, 2, 4, 8, 16, 32, 64) and grid * max(block // 64, 1) * rows >= n
