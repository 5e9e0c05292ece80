"""GPU parity of the fetch of many rows of five to seven chunks, which go to teams of four."""
import re

import numpy as np
import pytest
import torch

from test_gpu_fetch_teams import fetch_all, ibp  # noqa: F401
from test_gpu_wide import masks_of, rows_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,v,n", [(4, 513, 6143), (4, 513, 6144), (4, 640, 6150), (4, 895, 9001), (8, 321, 6200),
                                   (8, 448, 7001)])
def test_rows_of_five_to_seven_chunks(ibp, oracle, capfd, w, v, n):  # noqa: F811
    rng = np.random.default_rng(w * v + n)
    mask = masks_of("mixed", v, w, rng)
    bitval = rng.integers(0, 2 ** 63, size=v, dtype=np.uint64).astype(mask.dtype) & mask
    x = rows_for(211, mask, bitval, rng).view("i%d" % w)
    idx = rng.integers(0, 211, size=n)
    idx[[0, n - 1]] = [211, -1]
    print("small teams", w, v, n, flush=True)
    ibp.print_debug(True)
    try:
        capfd.readouterr()
        fetch_all(ibp, oracle, x, mask.view(x.dtype), bitval.view(x.dtype), idx)
        out = capfd.readouterr().out
    finally:
        ibp.print_debug(False)
    blocks = re.findall(r"team of waves per batch of rows, .* grid [0-9]+ x ([0-9]+),", out)
    assert blocks == [str(512 if n < 6144 else 256)] * 2
