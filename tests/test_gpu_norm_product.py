"""The norm of a few rows inside the product that reads them: the bits of the norm and the product one after the other."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows, outputs, width: a group of four waves with one to four rows, widths that end inside a pair of k-steps or in an even number of 16-byte chunks, outputs that end inside
# a unit, and each of the kernel's shapes
@pytest.mark.parametrize("M,N,K", [(1, 2304, 768), (2, 3072, 768), (3, 4096, 1024), (5, 2049, 776), (8, 2305, 1016), (7, 4096, 520), (6, 2320, 256),
                                   (1, 4097, 1024), (4, 8192, 1000), (5, 5000, 264), (8, 8191, 776), (2, 8200, 1024), (8, 11520, 1016)])
def test_norm_inside_the_product(M, N, K):
    from levanter_amd.kernels import get_kernels

    kern = get_kernels()
    assert kern.takes_norm(M, N, K)
    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    x, nw, nb, bias = rnd(M, K) * 3 + 1, 1 + 0.3 * rnd(K), 0.2 * rnd(K), rnd(N)
    w = (rnd(N, K) / K ** 0.5).bfloat16()
    kept = x.clone()
    for rms, shift, b, act in ((False, nb, bias, "gelu_new"), (True, None, None, "none"), (False, None, bias, "none"), (True, nb, None, "relu")):
        h = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
        kern.norm(x, nw, shift, 1e-5, h, rms=rms)
        want = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        kern.linear(h, w, b, want, activation=act)
        wide = torch.full((M, N + 16), float("nan"), dtype=torch.bfloat16, device=DEV)
        kern.linear_normed(x, nw, shift, 1e-5, rms, w, b, wide[:, :N], activation=act)
        assert torch.equal(wide[:, :N], want) and wide[:, N:].isnan().all() and torch.equal(x, kept)


def test_rows_that_are_not_finite_stay_alone():
    from levanter_amd.kernels import get_kernels

    kern = get_kernels()
    g = torch.Generator(device=DEV).manual_seed(0)
    M, N, K = 6, 4800, 1000
    x, nw, w = torch.randn(M, K, device=DEV, generator=g), torch.ones(K, device=DEV), torch.randn(N, K, device=DEV, generator=g).bfloat16()
    outs = []
    for bad in (None, float("inf"), float("nan")):
        y = x.clone()
        if bad is not None:
            y[2, K - 1] = bad
        outs.append(torch.empty(M, N, dtype=torch.bfloat16, device=DEV))
        kern.linear_normed(y, nw, None, 1e-5, False, w, None, outs[-1])
    others = [0, 1, 3, 4, 5]
    for o in outs[1:]:
        assert o[2].isnan().all() and torch.equal(o[others], outs[0][others])


def test_sizes_that_keep_the_two_kernels():
    from levanter_amd.kernels import KernelError, get_kernels

    kern = get_kernels()
    for M, N, K in ((9, 3072, 768), (8, 4800, 1032), (8, 768, 768), (8, 50257, 768)):
        assert not kern.takes_norm(M, N, K)
    x, w = torch.zeros(9, 768, device=DEV), torch.zeros(3072, 768, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(KernelError, match="no kernel"):
        kern.linear_normed(x, torch.ones(768, device=DEV), None, 1e-5, True, w, None, torch.empty(9, 3072, dtype=torch.bfloat16, device=DEV))


def test_a_forced_kernel_is_asked_anew():
    """The answer for a size goes by the kernel that takes its product, as the scratch memory does, and is forgotten with it."""
    from levanter_amd.kernels import KernelError, get_kernels

    kern = get_kernels()
    gemm = kern._unit("gemm_mfma")
    x, w, out = torch.ones(2, 768, device=DEV), torch.ones(3072, 768, dtype=torch.bfloat16, device=DEV), torch.empty(2, 3072, dtype=torch.bfloat16, device=DEV)
    args = (x, torch.ones(768, device=DEV), None, 1e-5, True, w, None, out)
    assert kern.takes_norm(2, 3072, 768)
    try:
        kern._check(gemm.lev_linear_mfma_force(2))
        kern._ws_need.clear()
        assert not kern.takes_norm(2, 3072, 768)
        with pytest.raises(KernelError, match="no kernel"):
            kern.linear_normed(*args)
    finally:
        kern._check(gemm.lev_linear_mfma_force(0))
        kern._ws_need.clear()
    assert kern.takes_norm(2, 3072, 768)
    kern.linear_normed(*args)
    assert bool((out.float() == 768).all())


# in float32: as above, widths that end inside a step of 16 and inside a wave's stretch of them, and sums too short for some of the waves
@pytest.mark.parametrize("M,N,K", [(3, 2304, 768), (4, 3072, 768), (8, 4096, 1024), (5, 1001, 772), (6, 640, 1020), (7, 2310, 516), (2, 4096, 1024), (8, 1024, 68), (4, 8192, 1000), (1, 6400, 512)])
def test_norm_inside_the_float32_product(M, N, K):
    from levanter_amd.kernels import get_kernels

    kern = get_kernels()
    assert kern.takes_norm_float32(M, N, K)
    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    x, nw, nb, bias, w = rnd(M, K) * 3 + 1, 1 + 0.3 * rnd(K), 0.2 * rnd(K), rnd(N), rnd(N, K) / K ** 0.5
    kept = x.clone()
    for rms, shift, b, act, pad in ((False, nb, bias, "gelu_new", 0), (True, None, None, "none", 3), (False, None, bias, "none", 16), (True, nb, None, "relu", 1)):
        h = torch.empty(M, K, device=DEV)
        kern.norm(x, nw, shift, 1e-5, h, rms=rms)
        want = torch.empty(M, N, device=DEV)
        kern.linear(h, w, b, want, activation=act)
        wide = torch.full((M, N + pad), float("nan"), device=DEV)
        kern.linear_normed(x, nw, shift, 1e-5, rms, w, b, wide[:, :N], activation=act)
        assert torch.equal(wide[:, :N], want) and wide[:, N:].isnan().all() and torch.equal(x, kept)
    x[M - 1, K - 1] = float("inf")
    out = torch.empty(M, N, device=DEV)
    kern.linear_normed(x, nw, nb, 1e-5, False, w, bias, out)
    assert out[M - 1].isnan().all() and not out[:M - 1].isnan().any()


def test_float32_weights_off_a_16_byte_boundary_keep_the_two_kernels():
    from levanter_amd.kernels import KernelError, get_kernels
    from levanter_amd.parts.base import BuildEnv
    from levanter_amd.parts.linear import Linear

    kern = get_kernels()
    env = BuildEnv(torch.float32, torch.device(DEV), kern)
    wide = torch.randn(1024 * 256 + 1, device=DEV)
    at, off = (Linear(wide[i:i + 1024 * 256].view(1024, 256), None, "out_in", env) for i in (0, 1))
    assert at.takes_norm(kern, 4) and not off.takes_norm(kern, 4)
    assert not any(kern.takes_norm_float32(*s) for s in ((9, 2304, 768), (4, 2304, 1028), (4, 2304, 770), (8, 8192, 1024), (1, 768, 768)))
    with pytest.raises(KernelError, match="aligned"):
        kern.linear_normed(torch.zeros(4, 256, device=DEV), torch.ones(256, device=DEV), None, 1e-5, True, off.weight, None, torch.empty(4, 1024, device=DEV))
