"""Prompt portions beside single tokens whose key ranges are split over the waves of the same launch's workgroups: as the two kernels one behind the other, bit for bit."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from levanter_amd.kernels import get_kernels

    return get_kernels()


@pytest.mark.parametrize("H,KVH,HD,PS,portions,singles,window", [
    (25, 25, 64, 16, [(256, 256)], [301, 150, 65, 64, 1] * 4, None),      # five ranges: one token and head a workgroup, three waves idle
    (25, 25, 64, 16, [(40, 90), (2, 2)], [128, 70], None),                # two: four a workgroup
    (12, 12, 64, 16, [(200, 200)], [190, 3, 129], None),                  # three: two, and two waves idle
    (16, 16, 128, 32, [(64, 300)], [250, 256, 17], None),                 # four: two
    (8, 8, 80, 16, [(33, 33)], [420, 500], 300),                          # eight under a window
    (32, 8, 64, 16, [(100, 100)], [300, 20, 260, 65], None),              # query heads that share keys
    (16, 1, 128, 16, [(100, 100)], [300, 20], None),                      # so many that the portions' keys have no room for the ranges: two launches
])
def test_split_ranges_beside_portions(K, H, KVH, HD, PS, portions, singles, window):
    from test_gpu_kernels import test_a_mixed_step_s_attention_equals_its_two_halves as halves

    halves(K, H, KVH, HD, PS, portions, singles, window)
