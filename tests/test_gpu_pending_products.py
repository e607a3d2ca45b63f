"""Products that leave their ranges to the pass that reads them: the passes' own tests, at their shapes with the kernel that splits the sum taken by force,
and at shapes that the rule gives to it."""
import pytest

import test_gpu_kelasun as kelasun
import test_gpu_lelatar as lelatar
import test_gpu_nakurax as nakurax

pytestmark = pytest.mark.gpu


@pytest.mark.usefixtures("splitting")
@pytest.mark.parametrize("M,N,Kd,bias", [(3, 512, 4096, True), (16, 512, 4096, False), (40, 264, 1024, True)])
def test_norm_behind_a_sum(M, N, Kd, bias):
    kelasun.test_the_norm_behind_a_sum_adds_up_a_product_that_has_left_its_ranges(M, N, Kd, bias)


@pytest.mark.usefixtures("splitting")
@pytest.mark.parametrize("M,N,Kd", [(3, 512, 4096), (16, 512, 4096), (40, 264, 1024)])
@pytest.mark.parametrize("plain_read", [True, False])
def test_group_norm(M, N, Kd, plain_read):
    lelatar.test_the_streams_pass_adds_up_a_product_that_has_left_its_ranges(M, N, Kd, plain_read)


@pytest.mark.usefixtures("splitting")
@pytest.mark.parametrize("M,N,Kd", [(8, 2048, 8192), (3, 1024, 4096), (64, 2048, 8192)])
def test_streams(M, N, Kd):
    nakurax.test_a_product_leaves_its_ranges_to_the_streams_pass(M, N, Kd)


@pytest.mark.parametrize("M,N,Kd", [(64, 1600, 6400), (64, 2048, 8192), (64, 4096, 16384)])
def test_the_rule_splits_long_sums_of_many_rows(M, N, Kd):
    from levanter_amd.kernels import get_kernels

    assert get_kernels()._unit("gemm_mfma").lev_linear_mfma_ranges(M, N, Kd) > 1
    skip = pytest.skip.Exception  # what the tests raise for a product without ranges
    try:
        kelasun.test_the_norm_behind_a_sum_adds_up_a_product_that_has_left_its_ranges(M, N, Kd, True)
        lelatar.test_the_streams_pass_adds_up_a_product_that_has_left_its_ranges(M, N, Kd, False)
        nakurax.test_a_product_leaves_its_ranges_to_the_streams_pass(M, N, Kd)
    except skip:
        pytest.fail("the product has left no ranges")
