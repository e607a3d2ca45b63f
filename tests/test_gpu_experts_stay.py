"""The experts' products by workgroups that stay on their CU and take several units in turn: rows that end inside a wave's 32, outputs that end inside a tile,
experts without rows, more tiles than a chiplet orders by size, several units a workgroup."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from levanter_amd.kernels import get_kernels

    return get_kernels()


EDGES = [1, 31, 0, 32, 33, 64, 65, 127, 128, 129, 260]


# sums from the shortest that goes this way (384: six k-tiles a unit); one workgroup has up to 1, 2, 7 and 40 units
@pytest.mark.parametrize("counts,Fo,Kd", [(EDGES * 20, 127, 384), (EDGES * 20, 63, 640), (EDGES * 8, 300, 512), ([200, 0, 5] * 4, 1601, 2048), ([97, 300, 0, 33] * 8, 776, 512), ([129] * 300, 200, 512),
                                          ([40] * 90, 1000, 768), ([129] * 300, 200, 384), ([5], 20000, 384), ([700, 3], 2600, 384)])
def test_against_float64(K, counts, Fo, Kd):
    from test_gpu_experts_many import _check

    assert K.lib.lev_moe_ring_takes(K.moe_max_tiles(sum(counts), len(counts), 128), Kd, 2 * Fo)  # with glu, most also without
    _check(K, counts, Fo, Kd, (Fo, Fo + 3) if Fo < 500 else (Fo,))


@pytest.mark.parametrize("counts,Fo,Kd", [(EDGES, 1, 512), (EDGES, 63, 640), ([200, 0, 5], 129, 2048), ([97, 300, 0, 33], 129, 384)])
def test_units_that_do_not_fill_the_chip(K, counts, Fo, Kd):
    """The tiles of 128 x 128 have them."""
    from test_gpu_experts_many import _check

    assert not K.lib.lev_moe_ring_takes(K.moe_max_tiles(sum(counts), len(counts), 128), Kd, 2 * Fo)
    _check(K, counts, Fo, Kd, (Fo, Fo + 3))
