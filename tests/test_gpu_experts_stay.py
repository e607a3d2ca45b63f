"""The experts' products by workgroups that stay on their CU and take several units in turn: rows that end inside a wave's 32, outputs that end inside a tile,
experts without rows, more tiles than a chiplet orders by size, several units a workgroup."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from levanter_amd.kernels import get_kernels

    return get_kernels()


# 384: the shortest sum that goes this way (six k-tiles a unit, a workgroup's only unit as long as the ring needs); one workgroup has up to 1, 2 and 7 units
@pytest.mark.parametrize("counts,Fo,Kd", [([1, 31, 0, 32, 33, 64, 65, 127, 128, 129, 260], 1, 512), ([1, 31, 0, 32, 33, 64, 65, 127, 128, 129, 260], 63, 640),
                                          ([200, 0, 5], 129, 2048), ([97, 300, 0, 33] * 8, 776, 512), ([129] * 300, 200, 512), ([40] * 90, 1000, 768),
                                          ([5], 40, 384), ([1, 31, 0, 32, 33, 64, 65, 127, 128, 129, 260], 63, 384), ([129] * 300, 200, 384)])
def test_against_float64(K, counts, Fo, Kd):
    from test_gpu_experts_many import _check

    _check(K, counts, Fo, Kd, (Fo, Fo + 3) if Fo < 500 else (Fo,))
