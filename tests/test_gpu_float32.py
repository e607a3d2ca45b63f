"""The 32-bit kernels on the GPU where their tiles, remainders and rules can go wrong, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
EPS = 2.0 ** -24


@pytest.fixture(scope="module")
def K():
    from levanter_amd.kernels import get_kernels

    return get_kernels()


def _rand(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


# rows, inputs, outputs: every tile of the list (rows x outputs of 16 x 16 .. 64 x 128), at its edges, one more and one less; inputs that are
# no multiple of a step of 16, fewer than the waves have steps, and (no multiple of 4) none that 16-byte loads take
LINEAR = [(1, 4, 1), (1, 64, 50), (3, 768, 768), (16, 100, 48), (17, 772, 33), (31, 1024, 130), (33, 20, 65), (64, 256, 4096), (65, 300, 1024), (129, 1028, 257),
          (203, 516, 1000), (400, 128, 1030), (777, 260, 1024), (1031, 96, 3000), (5, 6, 40), (70, 333, 129)]


@pytest.mark.parametrize("M,Ki,N", LINEAR)
@pytest.mark.parametrize("form", ["plain", "strided", "unaligned"])
def test_linear_float32(K, M, Ki, N, form):
    """Error bound: a sum of Ki products in any order is off by at most Ki * 2^-24 of the sum of their absolute values, bias and residual two roundings more."""
    pad, shift = {"plain": (0, 0), "strided": (8, 0), "unaligned": (3, 1)}[form]
    a_all = _rand(M * (Ki + pad) + shift, seed=1).to(DEV)
    a = a_all[shift:].view(M, Ki + pad)[:, :Ki]
    w, b = _rand(N, Ki, seed=2).to(DEV), _rand(N, seed=3).to(DEV)
    res = _rand(M, N, seed=4).to(DEV)
    want = a.double() @ w.double().T + b.double()
    size = a.double().abs() @ w.double().abs().T + b.double().abs()
    out_all = torch.full((M * (N + pad) + shift,), float("nan"), device=DEV)
    out = out_all[shift:].view(M, N + pad)[:, :N]
    K.linear(a, w, b, out)
    assert bool(((out.double() - want).abs() <= (Ki + 2) * EPS * size).all())
    assert int(torch.isnan(out_all).sum()) == M * pad + shift  # nothing beyond the output's own numbers
    out.copy_(res)
    K.linear(a, w, b, out, residual=out)
    assert bool(((out.double() - want - res.double()).abs() <= (Ki + 4) * EPS * (size + res.double().abs())).all())
    K.linear(a, w, b, out, activation="relu_squared", residual=res)
    assert bool(((out.double() - want.clamp(min=0) ** 2 - res.double()).abs() <= (2 * Ki + 8) * EPS * (size ** 2 + res.double().abs())).all())


def test_linear_float32_keeps_infinities_where_they_are(K):
    """An infinite input reaches the outputs of its own row only, also from the last, short step of a wave's inputs."""
    a, w = _rand(20, 52, seed=1).to(DEV), _rand(40, 52, seed=2).to(DEV)
    a[7, 51] = float("inf")
    out = torch.empty(20, 40, device=DEV)
    K.linear(a, w, None, out)
    want = a @ w.T
    assert torch.equal(torch.isinf(out), torch.isinf(want)) and not bool(torch.isnan(out).any())
    keep = [r for r in range(20) if r != 7]
    torch.testing.assert_close(out[keep], want[keep], rtol=1e-5, atol=52 * EPS * 50)
