"""GPU k-means at the ends of what it takes: 2^30 rows and more, and the least workspace."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ibp():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import invariantbitpacking_amd as m
    return m


# 512 threads per 128 rows, begun ones too: 2^32 - 512 are the most that a launch of tiles takes
@pytest.mark.parametrize("n", [(1 << 30) - 128, (1 << 30) - 127, (1 << 30) + 5])
def test_rows_beyond_one_launch_of_tiles(ibp, n):
    """2^30 rows of one column: four threads a row would be 2^32, more than a launch takes."""
    values = torch.tensor([0x0000ffff, 0x0000fff0, 0x7fff0000], dtype=torch.int32, device="cuda")
    x = values[(torch.arange(n, dtype=torch.int32, device="cuda") % 7 % 3).long()].view(n, 1)
    print("rows", n, flush=True)
    mask, bitval, cl = ibp.preprocess_kmeans(x, 2, seed=3)
    cl = cl.cuda()
    of = [cl[k::7] for k in range(7)]  # row i holds values[i % 7 % 3]
    first = [int(c[0]) for c in of]
    assert all(bool((c == f).all()) for c, f in zip(of, first))
    assert first[0] == first[3] == first[6] and first[1] == first[4] and first[2] == first[5]
    assert first[0] == first[1] != first[2]  # 4 bits apart; the third is 27 or more from both
    for c, rows in ((first[0], [0x0000ffff, 0x0000fff0]), (first[2], [0x7fff0000])):
        ones = rows[0] & rows[-1]
        zeros = ~rows[0] & ~rows[-1] & 0xffffffff
        assert int(mask[c, 0]) & 0xffffffff == ones | zeros
        assert int(bitval[c, 0]) & 0xffffffff == ones
