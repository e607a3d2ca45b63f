"""Products that leave their ranges to the pass that reads them: the passes' own tests at their shapes, with the kernel that splits the sum taken
by force. The rule gives some of these shapes to the kernel of few rows, which has nothing to leave, and the tests then end before the pass."""
import pytest

import test_gpu_kelasun as kelasun
import test_gpu_lelatar as lelatar
import test_gpu_nakurax as nakurax

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def splitting(monkeypatch):
    from levanter_amd.kernels import get_kernels

    K = get_kernels()
    gemm = K._unit("gemm_mfma")
    monkeypatch.setattr(K, "gemm_library", False)
    try:
        K._check(gemm.lev_linear_mfma_force(2))
        K._ws_need.clear()  # how much scratch memory a shape needs goes by the kernel that takes it
        yield
    finally:
        K._check(gemm.lev_linear_mfma_force(0))
        K._ws_need.clear()


@pytest.mark.parametrize("M,N,Kd,bias", [(3, 512, 4096, True), (16, 512, 4096, False), (40, 264, 1024, True)])
def test_norm_behind_a_sum(M, N, Kd, bias):
    kelasun.test_the_norm_behind_a_sum_adds_up_a_product_that_has_left_its_ranges(M, N, Kd, bias)


@pytest.mark.parametrize("M,N,Kd", [(3, 512, 4096), (16, 512, 4096), (40, 264, 1024)])
@pytest.mark.parametrize("plain_read", [True, False])
def test_group_norm(M, N, Kd, plain_read):
    lelatar.test_the_streams_pass_adds_up_a_product_that_has_left_its_ranges(M, N, Kd, plain_read)


@pytest.mark.parametrize("M,N,Kd", [(8, 2048, 8192), (3, 1024, 4096), (64, 2048, 8192)])
def test_streams(M, N, Kd):
    nakurax.test_a_product_leaves_its_ranges_to_the_streams_pass(M, N, Kd)
