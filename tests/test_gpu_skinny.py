"""The bfloat16 product of up to 64 rows at the edges of its launch shapes: columns that make half units, one to four units a workgroup and their
remainders, rows that fill one to four row tiles, inputs with a short last chunk and with fewer pairs than waves."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def K():
    from levanter_amd.kernels import get_kernels

    return get_kernels()


@pytest.mark.parametrize("N", [1, 7, 9, 2047, 2049, 4090, 4100, 8190, 8200, 11530, 12280, 12300, 16390])
@pytest.mark.parametrize("Ki", [8, 72, 200, 1784, 1800, 4168])
def test_linear_skinny_against_float64(K, N, Ki, monkeypatch):
    """bfloat16 operands are exact in float64; a sum of Ki products in 32 bits is off by at most Ki * 2^-24 of the sum of their absolute values."""
    gemm = K._unit("gemm_mfma")
    monkeypatch.setattr(K, "gemm_library", False)
    g = torch.Generator(device=DEV).manual_seed(N * 31 + Ki)
    w = torch.randn(N, Ki, device=DEV, generator=g).bfloat16()
    bias = torch.randn(N, device=DEV, generator=g)
    try:
        K._check(gemm.lev_linear_mfma_force(1))
        K._ws_need.clear()  # how much scratch memory a shape needs goes by the kernel that takes it
        for M in (1, 8, 9, 16, 17, 32, 33, 48, 49, 64):
            a = torch.randn(M, Ki + 8, device=DEV, generator=g).bfloat16()[:, :Ki]
            res = torch.randn(M, N, device=DEV, generator=g)
            want = a.double() @ w.double().T
            size = a.double().abs() @ w.double().abs().T
            out = torch.full((M, N + 3), float("nan"), device=DEV)
            K.linear(a, w, bias, out[:, :N], residual=res)
            err = (out[:, :N].double() - want - bias.double() - res.double()).abs()
            assert bool((err <= (Ki + 4) * 2.0 ** -24 * (size + bias.double().abs() + res.double().abs())).all()), M
            assert bool(torch.isnan(out[:, N:]).all())
            half = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
            K.linear(a, w, None, half)
            assert bool(((half.double() - want).abs() <= want.abs() * 2.0 ** -8 + Ki * 2.0 ** -24 * size).all()), M
    finally:
        K._check(gemm.lev_linear_mfma_force(0))
        K._ws_need.clear()


@pytest.mark.parametrize("N", [1, 24, 511, 768, 1024, 1025, 1600, 2048, 2049, 2304, 4096])
@pytest.mark.parametrize("Ki", [8, 72, 1600, 2040, 2048])
def test_linear_in_row_blocks_against_float64(K, N, Ki, monkeypatch):
    """65 to 256 rows of small weights, in blocks of 32 rows and columns where they make one round of the CUs, in the ring kernel beyond; the bound is the one above."""
    gemm = K._unit("gemm_mfma")
    monkeypatch.setattr(K, "gemm_library", False)
    g = torch.Generator(device=DEV).manual_seed(N * 31 + Ki)
    w = torch.randn(N, Ki, device=DEV, generator=g).bfloat16()
    bias = torch.randn(N, device=DEV, generator=g)
    for M in (65, 95, 128, 130, 193, 256):
        taken = -(-M // 32) * (-(-N // 256) * 8) <= 256
        assert (gemm.lev_linear_mfma_ring_of(M, N, Ki, 0) == -1) == taken
        assert not taken or gemm.lev_linear_mfma_ranges_of(M, N, Ki, 0) == 1
        a = torch.randn(M, Ki + 8, device=DEV, generator=g).bfloat16()[:, :Ki]
        res = torch.randn(M, N, device=DEV, generator=g)
        want = a.double() @ w.double().T + bias.double() + res.double()
        size = a.double().abs() @ w.double().abs().T + bias.double().abs() + res.double().abs()
        out = torch.full((M + 1, N + 3), float("nan"), device=DEV)
        K.linear(a, w, bias, out[:M, :N], residual=res)
        assert bool(((out[:M, :N].double() - want).abs() <= (Ki + 4) * 2.0 ** -24 * size).all()), M
        assert bool(torch.isnan(out[:M, N:]).all()) and bool(torch.isnan(out[M]).all())


@pytest.mark.parametrize("M,N,Ki,sums", [(8, 768, 3072, 16), (8, 4096, 4096, 16), (48, 4096, 4096, 16), (16, 2048, 8192, 16), (8, 6144, 6144, 16), (8, 4096, 16384, 16),
                                         (16, 12288, 4096, 16), (16, 50257, 768, 4), (16, 32000, 2048, 4)])
def test_the_sums_chains_of_roundings_stay_short(K, M, N, Ki, sums, monkeypatch):
    """Ki products in ``sums`` partial sums of n = Ki / 32 / sums instructions each, whose 32 products are added in four groups; the partial sums are then added in a
    row. After i of n equal steps a sum of random terms has i / n of its final variance, and each addition is off by 0.40 * 2^-24 of its result in root mean square
    (rounding to nearest, mantissas spread over their logarithm), so that the whole is off by that times sqrt((4 n + 1) / 2 + (sums + 1) / 2); 6 % more for
    the scatter over the outputs. Half as many sums would be 18 to 40 % above."""
    monkeypatch.setattr(K, "gemm_library", False)
    g = torch.Generator(device=DEV).manual_seed(N + Ki)
    a, w = torch.randn(M, Ki, device=DEV, generator=g).bfloat16(), torch.randn(N, Ki, device=DEV, generator=g).bfloat16()
    out = torch.empty(M, N, device=DEV)
    K.linear(a, w, None, out)
    want = a.double() @ w.double().T
    error = float((out.double() - want).norm() / want.norm())
    n = Ki / 32 / sums
    assert error <= 1.06 * 0.40 * 2.0 ** -24 * ((4 * n + 1) / 2 + (sums + 1) / 2) ** 0.5, error


@pytest.mark.parametrize("N", [40, 2500, 9000, 11536, 16400])
@pytest.mark.parametrize("pairs", [1, 2, 3, 4, 5, 6, 8, 9, 11, 12, 13, 17, 19, 33])
def test_linear_skinny_with_few_pairs_left(K, N, pairs, monkeypatch):
    """What is left of a sum behind the whole rounds of a workgroup's waves, for every number of it; every product once: ones give whole numbers, exactly."""
    gemm = K._unit("gemm_mfma")
    monkeypatch.setattr(K, "gemm_library", False)
    try:
        K._check(gemm.lev_linear_mfma_force(1))
        K._ws_need.clear()
        for Ki in (64 * pairs, 64 * pairs - 24):
            w = torch.ones(N, Ki, device=DEV, dtype=torch.bfloat16)
            w[:, Ki // 2] = 3.0
            for M in (1, 16, 17, 33, 64):
                a = torch.ones(M, Ki, device=DEV, dtype=torch.bfloat16)
                a[:, -1] = 5.0
                out = torch.full((M, N), float("nan"), device=DEV)
                K.linear(a, w, None, out)
                assert bool((out == (a[0].double() @ w[0].double()).item()).all()), (Ki, M)
    finally:
        K._check(gemm.lev_linear_mfma_force(0))
        K._ws_need.clear()


# Beyond the layers that the estimate was once fitted to: heads of some 50,000 outputs at a few and at 32 rows, long sums of a few hundred outputs, short sums
CHOICES = [(2, 59904, 1024), (25, 65024, 2048), (32, 50256, 2048), (22, 464, 16384), (25, 304, 11264), (9, 656, 16384), (58, 9696, 12992), (64, 3112, 128), (5, 1600, 256),
           (21, 6080, 256), (13, 50768, 256), (64, 34968, 1216)]


def test_the_choice_between_the_two_kernels_is_within_a_quarter_of_the_better_one(K):
    from test_gpu_kernels import _time_products

    gemm = K._unit("gemm_mfma")

    def timed(M, N, Ki, reps):
        weights = [torch.randn(N, Ki, device=DEV).bfloat16() for _ in range(max(3, min(12, int(6e8 / (N * Ki * 2)))))]
        a, bias, out = torch.randn(M, Ki, device=DEV).bfloat16(), torch.randn(N, device=DEV), torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        times = []
        for kind in (0, 1, 2):
            K._check(gemm.lev_linear_mfma_force(kind))
            K._ws_need.clear()
            times.append(_time_products(lambda w: K.linear(a, w, bias, out), weights, reps=reps))
        return times

    was, K.gemm_library = K.gemm_library, False
    try:
        report = [(c, timed(*c, 5)) for c in CHOICES]
        report = [(c, timed(*c, 15) if t[0] > 1.25 * min(t[1:]) else t) for c, t in report]  # over the line: once more, longer, before it counts
    finally:
        K.gemm_library = was
        K._check(gemm.lev_linear_mfma_force(0))
        K._ws_need.clear()
    assert not [x for x in report if x[1][0] > 1.25 * min(x[1][1:])], report


# beyond the ring kernel's sizes: 65 to 128 rows of more than 32,768 outputs (the kernel of streamed weights, all of a column's rows at once), more rows of four million outputs and more
# (tiles of 256 x 256, 256 x 192, 256 x 128 and 128 x 128, K in one range and in two and three)
BEYOND = [(65, 33001, 1608, 1), (100, 50257, 768, 1), (127, 32776, 4104, 1), (128, 40001, 200, 1), (512, 8192, 16384, 2), (385, 12288, 6400, 2), (700, 6400, 12288, 3), (257, 16390, 1032, 1),
          (2048, 6144, 72, 1), (513, 12289, 392, 1), (300, 22002, 1032, 1), (1300, 4004, 520, 1), (130, 33001, 264, 1), (4100, 1032, 72, 1)]


@pytest.mark.parametrize("M,N,Ki,ranges", BEYOND)
def test_products_beyond_the_ring_kernel(K, M, N, Ki, ranges, monkeypatch):
    """Every epilogue, outputs that end inside a tile, and sums whose ranges are left; the bound is the first test's."""
    gemm = K._unit("gemm_mfma")
    monkeypatch.setattr(K, "gemm_library", False)
    for left in (0, 1):
        assert gemm.lev_linear_mfma_ring_of(M, N, Ki, left) == -1 and gemm.lev_linear_mfma_ranges_of(M, N, Ki, left) == ranges
    g = torch.Generator(device=DEV).manual_seed(N + Ki)
    w = (torch.randn(N, Ki, device=DEV, generator=g) * Ki ** -0.5).bfloat16()
    a = torch.randn(M, Ki + 8, device=DEV, generator=g).bfloat16()[:, :Ki]
    bias, res = torch.randn(N, device=DEV, generator=g), torch.randn(M, N, device=DEV, generator=g)
    x, y = a.double(), w.double().T
    want, size = x @ y, x.abs() @ y.abs()
    bound = (Ki + 4) * 2.0 ** -24 * (size + bias.double().abs() + res.double().abs())
    out = torch.full((M, N + 3), float("nan"), device=DEV)
    K.linear(a, w, bias, out[:, :N], residual=res)
    assert bool(((out[:, :N].double() - want - bias.double() - res.double()).abs() <= bound).all()) and bool(torch.isnan(out[:, N:]).all())
    left = res.clone()
    pending = K.linear(a, w, bias, left, residual=left, may_leave_pending=True)
    assert (pending is not None) == (ranges > 1)
    if pending is not None:
        assert pending.n_ranges == ranges and torch.equal(left, res)
        K.finish(pending)
    assert bool(((left.double() - want - bias.double() - res.double()).abs() <= bound).all())
    half = torch.full((M, N), float("nan"), device=DEV, dtype=torch.bfloat16)
    for act, f in (("none", lambda u: u), ("gelu_new", lambda u: torch.nn.functional.gelu(u, approximate="tanh")), ("gelu", torch.nn.functional.gelu), ("silu", torch.nn.functional.silu)):
        K.linear(a, w, bias, half, activation=act)
        u = f(want + bias.double())
        assert float((half.double() - u).abs().max() / u.abs().max()) < 2e-2, act
