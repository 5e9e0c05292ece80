"""CPU tests of the k-means workspace: what a short one is refused with (before any GPU work)."""
import re

import pytest


@pytest.mark.parametrize("n,v,w,k", [(500, 2752, 8, 16), (16, 4096, 8, 2), (1, 1, 4, 1), (4096, 1024, 8, 16),
                                     (2449029, 50, 8, 4), (300, 21, 8, 24), (5000, 2752, 4, 16)])
def test_least_workspace_is_at_most_the_stated_one(n, v, w, k):
    from invariantbitpacking_amd import _capi
    full = _capi.lib().ibp_preprocess_kmeans_workspace_size(w, n, v, k)
    somewhere = 4096  # refused before it is used
    rc = _capi.lib().ibp_preprocess_kmeans_ws(w, somewhere, n, v, k, -1.0, 3, somewhere, somewhere, somewhere,
                                              somewhere, 256, None)
    assert rc == 1
    least = re.fullmatch(r"workspace too small \(256 < (\d+) bytes\)", _capi.last_error())
    assert least and int(least.group(1)) <= full
