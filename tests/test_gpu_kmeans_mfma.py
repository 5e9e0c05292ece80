"""GPU parity of preprocess_kmeans with up to 16 clusters (products of 0/1
matrices on the matrix units) at the edges of its tiles: 16-row tiles, 128-row
blocks, steps of 16 dwords, one, four and sixteen waves per tile, row parts,
rows whose bit sums pass an accumulator's exact range, workspaces with and
without room for the bit planes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ibp():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import invariantbitpacking_amd as m
    return m


def groups(n, v, w, k, seed):
    """Rows around k random centres (some columns shared), a few of them far off."""
    rng = np.random.default_rng(seed)
    dt = np.dtype("u%d" % w)
    centres = rng.integers(0, 256, size=(k, v * w), dtype=np.uint8)
    x = centres[rng.integers(0, k, size=n)]
    x ^= (1 << rng.integers(0, 8, size=x.shape, dtype=np.uint8)) * (rng.random(x.shape) < 0.1).astype(np.uint8)
    x[::11] = rng.integers(0, 256, size=x[::11].shape, dtype=np.uint8)
    return np.ascontiguousarray(x).view(dt).view("i%d" % w)


def check(ibp, oracle, x, k, where="device"):
    om, ob, oc = oracle.kmeans(x, k, seed=3)[:3]
    t = torch.from_numpy(x).cuda() if where == "device" else torch.from_numpy(x).pin_memory()
    m, b, c = ibp.preprocess_kmeans(t, k, seed=3)
    assert np.array_equal(c.numpy(), oc)
    assert np.array_equal(m.cpu().numpy().view(om.dtype).reshape(om.shape), om)
    assert np.array_equal(b.cpu().numpy().view(ob.dtype).reshape(ob.shape), ob)


@pytest.mark.parametrize("n,v,w,k", [(1, 1, 4, 1), (3, 5, 8, 16), (15, 16, 4, 2), (16, 17, 4, 16), (17, 8, 8, 3),
                                     (127, 33, 4, 7), (128, 40, 8, 16), (129, 9, 8, 15), (700, 64, 8, 16),
                                     (4100, 2, 4, 5), (9000, 15, 8, 16), (2100, 300, 4, 16), (900, 515, 8, 11),
                                     (33000, 70, 4, 4)])
def test_kmeans_up_to_16_matches_oracle(ibp, oracle, n, v, w, k):
    check(ibp, oracle, groups(n, v, w, max(k, 2), seed=n + v), k)


def test_kmeans_rows_of_2_mib(ibp, oracle):
    """2^24 bits and more per row: sixteen waves share a row's sum."""
    check(ibp, oracle, groups(37, 270001, 8, 3, seed=1), 3)


def test_kmeans_table_in_row_parts(ibp, oracle):
    """A narrow table of many rows: its rows are cut into parts that add up."""
    check(ibp, oracle, groups(700001, 50, 8, 3, seed=2), 2)


@pytest.mark.parametrize("n,v,w,k", [(1, 1, 4, 1), (129, 9, 8, 15), (5000, 37, 4, 6), (300, 21, 8, 24), (0, 3, 4, 2)])
def test_kmeans_workspaces(ibp, oracle, n, v, w, k):
    """The stated size, the library's own memory, and less down to what the
    call refuses: every call that runs gives the oracle's result."""
    from invariantbitpacking_amd import _capi
    x = groups(n, v, w, max(k, 2), seed=n + v) if n else np.zeros((0, v), "i%d" % w)
    om, ob, oc = oracle.kmeans(x, k, seed=3)[:3]
    t = torch.from_numpy(x).cuda()
    full = _capi.lib().ibp_preprocess_kmeans_workspace_size(w, n, v, k)
    assert full > 0 and _capi.lib().ibp_preprocess_kmeans_workspace_size(3, n, v, k) == 0
    ran = []
    for size in [None, full] + [full * i // 16 for i in range(15, 0, -1)] + [256]:
        m = torch.full((k, v), 5, dtype=t.dtype, device="cuda")
        b = torch.full((k, v), 5, dtype=t.dtype, device="cuda")
        c = torch.full((max(n, 1),), -1, dtype=torch.int32, device="cuda")
        ws = torch.empty((size or 0) + 1, dtype=torch.uint8, device="cuda")
        rc = _capi.lib().ibp_preprocess_kmeans_ws(w, t.data_ptr(), n, v, k, -1.0, 3, m.data_ptr(), b.data_ptr(),
                                                  c.data_ptr(), ws.data_ptr() if size else None, size or 0,
                                                  torch.cuda.current_stream().cuda_stream)
        ran.append(rc == 0)
        if rc:
            continue
        assert np.array_equal(c.cpu().numpy()[:n], oc)
        assert np.array_equal(m.cpu().numpy().view(om.dtype).reshape(om.shape), om)
        assert np.array_equal(b.cpu().numpy().view(ob.dtype).reshape(ob.shape), ob)
    assert ran[0] and ran[1] and not ran[-1]
    assert ran[1:] == sorted(ran[1:], reverse=True)
