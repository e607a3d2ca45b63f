"""Which parts are given rows that their first product normalises itself, and what becomes of such rows in a product that does more than read them: on the CPU, with plain
kernels that say they take every norm along."""
import torch

from emulated_kernels import EmulatedKernels
from levanter_amd.kernels.library import KernelError
from levanter_amd.parts.base import BuildEnv, StepContext
from levanter_amd.parts.block import PreNormBlock
from levanter_amd.parts.feed_forward import DenseMlp, GatedMlp
from levanter_amd.parts.linear import Linear, RowsAhead
from levanter_amd.parts.norm import LayerNorm
from levanter_amd.parts.spec import PartSpec

T, D, F = 3, 16, 32


class TakesNorms(EmulatedKernels):
    widths = (F, 2 * F)

    def __init__(self):
        self.taken = 0

    def takes_norm(self, M, N, K):
        return N in self.widths

    def linear_normed(self, x, norm_weight, norm_bias, eps, rms, w, bias, out, activation="none"):
        if w.shape[0] not in self.widths or out.dtype != torch.bfloat16 or x.data_ptr() % 16 or not x.is_contiguous():
            raise KernelError("norm and linear: no kernel")
        self.taken += 1
        h = torch.empty_like(x, dtype=torch.bfloat16)
        self.norm(x, norm_weight, norm_bias, eps, h, rms=rms)
        self.linear(h, w, bias, out, activation=activation)


def _parts(norm=LayerNorm, mlp=DenseMlp):
    g = torch.Generator().manual_seed(0)
    env = BuildEnv(torch.bfloat16, torch.device("cpu"), TakesNorms())
    ctx = StepContext(kernels=env.kernels, dtype=env.dtype, device=env.device, n_tokens=T, tokens=None, attention=None, seq_slots=None, host={})
    n = norm(PartSpec("layernorm", dict(dim=D, eps=1e-5)), {"weight": torch.randn(D, generator=g), "bias": torch.randn(D, generator=g)}, env)
    names = ("gate.weight", "up.weight") if issubclass(mlp, GatedMlp) else ("up.weight",)
    tensors = {"down.weight": torch.randn(D, F, generator=g), **{k: torch.randn(F, D, generator=g) for k in names}}
    m = mlp(PartSpec("mlp", dict(dim=D, inner_dim=F, activation="silu")), tensors, env)
    return n, m, ctx, env.kernels, torch.randn(T, D, generator=g)


def _run(norm, mlp, x, ctx):
    x = x.clone()
    mlp.forward(PreNormBlock._normed(norm, mlp, x, ctx), x, ctx)
    return x


def _check(norm, mlp, ctx, kernels, x, taken):
    want = x.clone()
    mlp.forward(norm(want, ctx), want, ctx)
    assert torch.equal(_run(norm, mlp, x, ctx), want) and kernels.taken == taken


def test_parts_as_they_are():
    for mlp in (DenseMlp, GatedMlp):
        _check(*(p := _parts(mlp=mlp))[:4], p[4], taken=1)


def test_a_part_that_reads_its_rows_elsewhere_gets_rows():
    class Reads(DenseMlp):
        def forward(self, h, x, ctx):
            x += h.float() * 0.5
            super().forward(h, x, ctx)

    class Inner(GatedMlp):
        def _inner(self, h, ctx):
            return super()._inner(h * 2, ctx)

    for mlp in (Reads, Inner):
        _check(*(p := _parts(mlp=mlp))[:4], p[4], taken=0)
    n, m, ctx, k, x = _parts()
    own, seen = m.forward, []
    m.forward = lambda h, x, ctx: (seen.append(h), own(h, x, ctx))
    _check(n, m, ctx, k, x, taken=0)
    assert all(isinstance(h, torch.Tensor) for h in seen)


def test_a_norm_of_its_own_is_not_passed_by():
    class Scaled(LayerNorm):
        def __call__(self, x, ctx, rows=None):
            return super().__call__(x, ctx, rows) * 2

    _check(*(p := _parts(norm=Scaled))[:4], p[4], taken=0)


def test_another_product_in_the_linears_place():
    n, m, ctx, k, x = _parts()
    up = m.up
    m.up = lambda h, ctx, **args: up(h, ctx, **args) + 1
    _check(n, m, ctx, k, x, taken=0)


def test_rows_that_the_kernel_cannot_read():
    n, m, ctx, k, x = _parts()
    storage = torch.empty(T * D + 1)
    odd = storage[1:].view(T, D).copy_(x)
    assert isinstance(PreNormBlock._normed(n, m, odd, ctx), torch.Tensor)
    assert isinstance(PreNormBlock._normed(n, m, torch.empty(D, T).t().copy_(x), ctx), torch.Tensor)


def test_a_product_that_does_more_than_the_kernel_makes_the_rows_first():
    n, m, ctx, k, x = _parts()
    rows = RowsAhead(x, n)
    h = n(x, ctx)
    narrow = Linear(m.up.weight[:24], None, "out_in", BuildEnv(torch.bfloat16, torch.device("cpu"), k))
    res = torch.randn(T, F)
    for product, args in ((m.up, dict(residual=res.clone(), final=True)), (m.up, dict(out=torch.empty(T, F), may_leave=True)), (m.up, dict(out_dtype=torch.float32)), (narrow, {})):
        fresh = lambda: {a: v.clone() if isinstance(v, torch.Tensor) else v for a, v in args.items()}
        assert torch.equal(product(rows, ctx, **fresh()), product(h, ctx, **fresh())), args
    assert k.taken == 0
    assert torch.equal(m.up(rows, ctx), m.up(h, ctx)) and k.taken == 1
