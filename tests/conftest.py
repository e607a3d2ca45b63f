import os
import sys

import pytest

_HERE = os.path.dirname(os.path.abspath(__file__))
_ROOT = os.path.dirname(_HERE)
for p in (_HERE, _ROOT):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture
def splitting(monkeypatch):
    """Products go to the kernel that splits the sum over K, whatever the rule of a shape."""
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


# tests of the passes that add up unsummed products: the rule gives some of their small shapes to the kernel of few rows, which has nothing to leave
LEFT_RANGES = {"test_the_norm_behind_a_sum_adds_up_a_product_that_has_left_its_ranges", "test_the_streams_pass_adds_up_a_product_that_has_left_its_ranges",
               "test_a_product_leaves_its_ranges_to_the_streams_pass"}


@pytest.fixture(autouse=True)
def ranges_are_left(request):
    if getattr(request.node, "originalname", None) in LEFT_RANGES:
        request.getfixturevalue("splitting")
