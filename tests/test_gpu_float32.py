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


# rows, inputs, outputs: every tile whose operands come straight from memory (16 x 16 .. 32 x 64 here, 64 x 64 at the end), at its edges, one more and one less; inputs
# that are no multiple of a step of 16, fewer than the waves have steps, and (no multiple of 4) none that 16-byte loads take. (13, 264, 50257) takes
# 16 x 32 and (15, 264, 11531) 16 x 64. That all kernels are among them is a test below.
LINEAR = [(1, 4, 1), (1, 64, 50), (3, 768, 768), (16, 100, 48), (17, 772, 33), (31, 1024, 130), (33, 20, 65), (64, 256, 4096), (65, 300, 1024), (129, 1028, 257),
          (203, 516, 1000), (400, 128, 1030), (777, 260, 1024), (1031, 96, 3000), (15, 264, 11531), (13, 264, 50257), (5, 6, 40), (70, 333, 129)]
# the tiles whose operands come through LDS (32 x 32, 32 x 64, 32 x 96, 64 x 64, 64 x 96): ends inside a tile, K of one step, with a short one, of
# odd and even numbers of steps, of pieces of 128 and 256 and one step more; and tiles of split operands (more below)
LINEAR += [(404, 768, 3072), (289, 100, 2051), (1031, 32, 3001), (801, 1028, 1030), (777, 300, 3072), (2047, 292, 4097), (609, 516, 2310), (2047, 260, 2310),
           (1000, 260, 4097), (1030, 1028, 4100), (2047, 516, 3071), (1153, 284, 1602), (1153, 284, 2303), (511, 412, 3202), (1353, 276, 2199), (447, 1060, 3454),
           (1406, 1252, 961), (1665, 1236, 863), (777, 1028, 4100)]
# up to eight rows and four outputs a workgroup: 1, 2, 4 and 8 rows' room full and not, outputs that end inside a workgroup, K of less than a thread each,
# one stretch of 2,048, two, a short one more; and shapes that the rule gives to the tiles
LINEAR += [(1, 8196, 64), (2, 1028, 3001), (3, 4100, 130), (4, 2048, 1601), (5, 2052, 33), (8, 1024, 777), (7, 4096, 1600), (8, 1020, 40), (4, 1600, 1601), (1, 100, 6401)]

# 64 x 64 straight from memory: rows and outputs that end inside a tile, K with a short last step (of 256 inputs and more the tiles of split operands have these)
LINEAR += [(935, 228, 8317), (129, 3396, 4949), (195, 3364, 3558), (777, 4100, 1030)]


def _kernel(K, M, Ki, N):
    """Which kernel runs a product of aligned rows: "split" and the tile, or the place of the 32-bit instruction's kernel."""
    split = K.lib.lev_linear_f32_split(M, N, Ki)
    return ("split", split) if split >= 0 else K.lib.lev_linear_f32_choice(M, N, Ki)


def test_every_kernel_is_among_the_shapes(K):
    """Room for 8, 4, 2 and 1 rows (-8 .. -1), seven tiles straight from memory, five through LDS, three of split operands."""
    assert {_kernel(K, *s) for s in LINEAR if s[1] % 4 == 0} == {-8, -4, -2, -1, *range(12), ("split", 0), ("split", 1), ("split", 2)}


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


@pytest.mark.parametrize("M,N,Ki", [(2048, 4096, 64), (1024, 3072, 96), (1024, 3072, 128), (2048, 4096, 128), (2048, 2304, 192), (777, 2304, 256), (404, 4096, 384),
                                    (777, 2304, 384), (777, 1024, 512), (777, 1024, 1024)])
def test_short_sums_are_no_long_chains(K, M, N, Ki):
    """Relative error in the 2-norm of products of normal numbers. A rounding is off by 0.42 * 2^-24 of its result (2^-23 / sqrt(12), times the root mean square of
    1 / x over a power of two); the sums in a chain of c of the K numbers are j / K of the whole's square, j = 1 .. c: chains of c and their K / c joins make
    0.42 * 2^-24 * sqrt(c / 2 + K / (2 c)). Chains: a quarter of K in steps of 16, at most 128; 15 % for what is drawn and for products of 4 at a time."""
    a, w = _rand(M, Ki, seed=1).to(DEV), _rand(N, Ki, seed=2).to(DEV)
    out = torch.empty(M, N, device=DEV)
    K.linear(a, w, None, out)
    want = a.double() @ w.double().T
    c = min(128, -(-Ki // 64) * 16)
    assert float((out.double() - want).norm() / want.norm()) <= 1.15 * 0.42 * EPS * (c / 2 + Ki / (2 * c)) ** 0.5


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


@pytest.mark.parametrize("kernel,M,Ki,N", [(7, 289, 100, 2051), (9, 609, 516, 2310), (10, 1153, 284, 2303), (11, 1406, 1252, 961), (6, 935, 228, 8317), (-1, 1, 8196, 64), (-4, 3, 4100, 130), (-8, 8, 1028, 777),
                                           (11, 1030, 1028, 4100), (("split", 1), 513, 516, 6530), (("split", 2), 129, 3396, 4949)])
def test_linear_float32_keeps_infinities_where_they_are_in_every_kernel(K, kernel, M, Ki, N):
    """Tiles through LDS with a short step of one, two and four sums, 64 x 64 straight from memory, rooms for 1, 4 and 8 rows whose last stretch is short, and tiles of split operands: an infinite
    last input reaches its own row, an infinite last weight its own output, and nothing else is anything but finite."""
    assert _kernel(K, M, Ki, N) == kernel
    a, w = _rand(M, Ki, seed=1).to(DEV), _rand(N, Ki, seed=2).to(DEV)
    row, col = M // 2, N // 2
    a[row, Ki - 1] = float("inf")
    w[col, Ki - 1] = float("-inf")
    out = torch.empty(M, N, device=DEV)
    K.linear(a, w, None, out)
    want = torch.zeros(M, N, dtype=torch.bool, device=DEV)
    want[row] = want[:, col] = True
    assert torch.equal(torch.isinf(out), want) and not bool(torch.isnan(out).any())
    assert torch.equal(out[row] > 0, w[:, Ki - 1] > 0)


# products whose operands are split into bfloat16 numbers: tiles of 128 x 128, 64 x 128 and 64 x 64 outputs that end inside a tile, whole steps of 32 inputs, a partial one of 4 and of 28,
# odd and even numbers of steps, numbers that the two groups of a 64 x 64 tile share unevenly, sums that are joined once and often, and long ones
SPLIT = [(0, 1025, 260, 3457), (0, 511, 284, 7171), (0, 1151, 288, 3326), (0, 1153, 4100, 2053), (1, 514, 256, 6404), (1, 1410, 256, 8325), (1, 513, 516, 6530), (1, 385, 540, 8831), (1, 385, 284, 4476),
         (2, 321, 1028, 2244), (2, 127, 1052, 6204), (2, 65, 3396, 5503), (2, 193, 1316, 3582), (2, 66, 4100, 5566), (2, 770, 2052, 961)]


@pytest.mark.parametrize("tile,M,Ki,N", SPLIT)
def test_split_products(K, tile, M, Ki, N):
    """Bound: Ki roundings, at most, of what has been added up so far, and at most 2^-23 of every product for the parts that are left out; bias and residual two more."""
    assert K.lib.lev_linear_f32_split(M, N, Ki) == tile
    a_all, w, b, res = _rand(M, Ki + 8, seed=1).to(DEV), _rand(N, Ki, seed=2).to(DEV), _rand(N, seed=3).to(DEV), _rand(M, N, seed=4).to(DEV)
    a = a_all[:, :Ki]
    want = a.double() @ w.double().T + b.double()
    size = a.double().abs() @ w.double().abs().T + b.double().abs()
    out = torch.full((M, N + 3), float("nan"), device=DEV)
    K.linear(a, w, b, out[:, :N], residual=res)
    assert bool(((out[:, :N].double() - want - res.double()).abs() <= (Ki + 6) * EPS * (size + res.double().abs())).all())
    assert bool(torch.isnan(out[:, N:]).all())
    got = torch.empty(M, N, device=DEV)
    K.linear(a, w, None, got)
    exact = a.double() @ w.double().T
    # in the 2-norm as below, with sums of their own for at most 256 numbers: 0.42 * 2^-24 * sqrt(c / 2 + K / (2 c)), c = 128
    assert float((got.double() - exact).norm() / exact.norm()) <= 1.15 * 0.42 * EPS * (64 + Ki / 256) ** 0.5


@pytest.mark.parametrize("tile,M,Ki,N", [(0, 511, 284, 7171), (1, 513, 516, 6530), (2, 193, 1316, 3582)])
def test_split_products_of_the_smallest_and_largest_numbers(K, tile, M, Ki, N):
    """Powers of two on the operands change nothing, down to numbers whose last bits are the smallest there are and up to the largest, which have no bfloat16 parts."""
    assert K.lib.lev_linear_f32_split(M, N, Ki) == tile
    a, w = _rand(M, Ki, seed=1).to(DEV), _rand(N, Ki, seed=2).to(DEV)
    a = a.sign() * a.abs().clamp(min=2.0 ** -6)
    exact = a.double() @ w.double().T
    for up, other in ((-119, 40), (119, -60), (60, -60)):
        got = torch.empty(M, N, device=DEV)
        K.linear(a * 2.0 ** up, w * 2.0 ** other, None, got)
        assert float((got.double() * 2.0 ** -(up + other) - exact).norm() / exact.norm()) <= 1.15 * 0.42 * EPS * (64 + Ki / 256) ** 0.5
    a[M // 2, 5], w[N // 2, 7] = 3.4e38, float("nan")
    a[3, Ki - 1] = float("-inf")
    a[M - 1, 0], w[0, 0] = 0.0, float("inf")
    got = torch.empty(M, N, device=DEV)
    K.linear(a, w, None, got)
    want = (a.double() @ w.double().T).float()  # the same places beyond the range of 32 bits
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    inf = torch.isinf(want)
    assert torch.equal(got[inf] > 0, want[inf] > 0)
    size = (a.double().abs() @ w.double().abs().T)
    fine = ~inf & ~torch.isnan(want)
    assert bool(((got.double() - want.double()).abs() <= (Ki + 6) * EPS * size)[fine].all())


@pytest.mark.parametrize("tile,M,Ki,N", [(0, 511, 284, 7171), (1, 513, 516, 6530), (2, 193, 1316, 3582)])
@pytest.mark.parametrize("terms", [1, 2])
def test_split_products_of_a_few_terms(K, tile, M, Ki, N, terms):
    """Rows with one and two inputs that are not zero, where no long sum hides a product's own error. Of numbers in [1, 2) the second and third bfloat16 parts are at most 2^-8 and 2^-17,
    so that the three partial products left out are at most 2^-24 + 2^-34 of a product; the sums' roundings are one for each term and, of the other parts (2^-7), an eighth in all."""
    assert K.lib.lev_linear_f32_split(M, N, Ki) == tile
    g = torch.Generator().manual_seed(tile)
    at = torch.stack([torch.randperm(Ki, generator=g)[:terms] for _ in range(M)])
    a = torch.zeros(M, Ki).scatter_(1, at, (1 + torch.rand(M, terms, generator=g)) * 2.0 ** torch.randint(-20, 20, (M, terms), generator=g)).to(DEV)
    w = ((1 + torch.rand(N, Ki, generator=g)) * (torch.randint(0, 2, (N, Ki), generator=g) * 2 - 1)).to(DEV)
    got = torch.empty(M, N, device=DEV)
    K.linear(a, w, None, got)
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    assert bool(((got.double() - want).abs() <= (1 + terms + 0.125) * EPS * size).all())


@pytest.mark.parametrize("choice,M,Ki,N", [(8, 273, 772, 9001), (9, 129, 516, 9001), (10, 177, 516, 9001), (11, 465, 256, 9001)])
def test_rows_too_far_apart_to_be_split(K, choice, M, Ki, N):
    """Rows more than 2^22 numbers apart: the tiles through LDS on the 32-bit instruction."""
    assert K.lib.lev_linear_f32_choice(M, N, Ki) == choice
    far = 2 ** 22 + 4
    a = torch.empty(M * far, device=DEV).as_strided((M, Ki), (far, 1))
    a.copy_(_rand(M, Ki, seed=1))
    w, b, res = _rand(N, Ki, seed=2).to(DEV), _rand(N, seed=3).to(DEV), _rand(M, N, seed=4).to(DEV)
    out = torch.empty(M, N, device=DEV)
    K.linear(a, w, b, out, residual=res)
    want = a.double() @ w.double().T + b.double() + res.double()
    size = a.double().abs() @ w.double().abs().T + b.double().abs() + res.double().abs()
    assert bool(((out.double() - want).abs() <= (Ki + 4) * EPS * size).all())


def test_a_waves_sum_is_the_tree_over_lane_numbers(K):
    """Every lane's number is exact (one of four inputs counts), so that the sums are those of the 64 lanes, halves first, then of neighbours 16, 8, 4, 2 and 1 apart, and of the
    eight waves in order, bit by bit."""
    a = torch.randn(1, 2048, generator=torch.Generator().manual_seed(1)) * torch.logspace(-3, 3, 2048)
    w = torch.zeros(64, 2048)
    for n in range(64):
        w[n, n % 4::4] = 1.0
    assert K.lib.lev_linear_f32_choice(1, 64, 2048) == -1
    out = torch.empty(1, 64, device=DEV)
    K.linear(a.to(DEV), w.to(DEV), None, out)
    for n in range(4):
        v = a[0, n::4].reshape(8, 64)
        for apart in (32, 16, 8, 4, 2, 1):
            v = v + v[:, torch.arange(64) ^ apart]
        total = torch.zeros(())
        for part in v[:, 0]:
            total = total + part
        assert bool((out[0, n::4].cpu() == total).all())


def _attention_float64(q, kp, vp, bt, runs, H, KVH, HD, PS, scale, window):
    """Whole sequences from the pages in float64; only what a query sees is read."""
    out, t = [], 0
    for s, (n, kv) in enumerate(runs):
        pages = bt[s, :(kv + PS - 1) // PS].long()
        k = kp.view(-1, KVH, HD // 8, PS, 8)[pages].permute(1, 0, 3, 2, 4).reshape(KVH, -1, HD)[:, :kv].double()
        v = vp.view(-1, KVH, HD, PS)[pages].permute(1, 0, 3, 2).reshape(KVH, -1, HD)[:, :kv].double()
        for i in range(n):
            pos = kv - n + i
            lo = max(0, pos - window + 1) if window else 0
            for h in range(H):
                w = torch.softmax(k[h * KVH // H, lo:pos + 1] @ q[t, h * HD:(h + 1) * HD].double() * scale, 0)
                out.append(w @ v[h * KVH // H, lo:pos + 1])
            t += 1
    return torch.stack(out).view(t, H * HD)


# runs of (tokens, keys after the step): tiles of 16 rows with 1 to 16 in use, blocks of 64 and 32 keys at their edges, single tokens beside
# them; groups of heads that fill a column set, more and less; every head size; single tokens that need more than 64 KB of LDS (the last two)
ATTENTION = [(4, 4, 64, 16, [(2, 2), (17, 17), (1, 64), (1, 65), (15, 80)], None), (16, 1, 16, 16, [(1, 1), (1, 33), (3, 130)], None),
             (20, 1, 32, 32, [(1, 257), (18, 18)], 20), (6, 2, 48, 16, [(1, 300), (129, 140)], 64), (5, 5, 80, 48, [(33, 97), (1, 31)], None),
             (3, 1, 96, 16, [(1, 128), (16, 16)], 17), (2, 2, 112, 64, [(1, 127), (31, 31)], None), (8, 4, 128, 16, [(1, 513), (40, 72), (1, 2)], 1),
             (16, 1, 128, 16, [(1, 300), (1, 16), (20, 20), (1, 1)], None), (32, 2, 112, 32, [(1, 200), (1, 33)], 100)]


@pytest.mark.parametrize("H,KVH,HD,PS,runs,window", ATTENTION)
def test_attention_float32(K, H, KVH, HD, PS, runs, window):
    """Weights are off by the scores' rounding, HD * 2^-24 of |q| |k| * scale (about 40 here) and a few units of the exponential: 2e-5 of the values."""
    from helpers import make_meta
    from test_gpu_kernels import _fill_cache

    kv = [k for _, k in runs]
    bt, kp, vp, kd, vd, _, _ = _fill_cache(K, torch.float32, kv, KVH, HD, PS, sum((k + PS - 1) // PS for k in kv) + 3, seed=5)
    T = sum(n for n, _ in runs)
    q = _rand(T, H * HD + 4, seed=6)
    want = _attention_float64(q, kp, vp, bt, runs, H, KVH, HD, PS, HD ** -0.5, window)
    for shift in (0, 1):  # the second time nothing is aligned: the plain kernel
        qd = torch.empty(T * (H * HD + 4) + shift, device=DEV)[shift:].view(T, H * HD + 4)
        qd.copy_(q)
        got = torch.full((T, H * HD), float("nan"), device=DEV)
        K.paged_attention(qd[:, :H * HD], got, kd, vd, make_meta(runs, DEV), n_heads=H, n_kv_heads=KVH, head_dim=HD, page_size=PS, scale=HD ** -0.5,
                          window=window, block_tables=bt.to(DEV))
        torch.testing.assert_close(got.cpu().double(), want, rtol=2e-5, atol=2e-5)


# runs in workgroups of four waves: more than 384 of them (tiles x 8 x heads) at every head size; key ranges that end and begin inside, at and behind a wave's block of 16
@pytest.mark.parametrize("HD", range(16, 129, 16))
@pytest.mark.parametrize("window", [None, 33])
def test_attention_float32_of_many_heads(K, HD, window):
    test_attention_float32(K, 32, 8, HD, 16, [(15, 63), (33, 64), (17, 81), (1, 40)], window)


# the same over many rounds of the waves
@pytest.mark.parametrize("HD", [16, 64, 128])
@pytest.mark.parametrize("window", [None, 333])
def test_attention_float32_of_many_heads_over_long_contexts(K, HD, window):
    test_attention_float32(K, 64, 8, HD, 16, [(18, 611), (2, 1030), (1, 700)], window)


# single tokens in workgroups of four waves (head sizes up to 96): more than 256 of them (tokens x key/value heads); key ranges of less than a wave's block of 32 keys to several rounds
@pytest.mark.parametrize("HD", range(16, 97, 16))
@pytest.mark.parametrize("window", [None, 50])
def test_attention_float32_of_many_single_tokens(K, HD, window):
    test_attention_float32(K, 16, 16, HD, 16, [(1, n) for n in (1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 160, 161, 255, 300)], window)


# the kernels of runs with four and eight waves, of single tokens with four and eight; (rows of) requests, heads
@pytest.mark.parametrize("runs,H,bound", [([64], 64, 1.6), ([17], 16, 1.4), ([1] * 260, 16, 1.3), ([1] * 60, 16, 1.3)])
@pytest.mark.parametrize("HD", [64, 128])
def test_attention_float32_denominators_of_long_contexts(K, runs, H, bound, HD):
    """Scores are exact, the only value is the first key's, whose weight is 1 throughout: an output is 1 / the sum of 16,384 weights. Its error is the exponentials' and
    the merge's, about one unit of 2^-24, and that of the chain of sums: each lane's of every fourth four keys of a wave's, of n additions, 0.3 sqrt(n / 3) / 2 units.
    (Measured 1.3, 1.1, 1.1, 1.1; a sum over a block's lanes that joins one over the context: 2.1, 1.5, 1.6, 1.4.)"""
    from helpers import make_meta

    n, PS = 16384, 16
    g = torch.Generator().manual_seed(3)
    x = torch.clamp(torch.round(torch.randn(n, HD, generator=g) * 16) / 16, max=4.0)
    x[0] = 4.0
    kd = x.view(n // PS, PS, HD // 8, 8).permute(0, 2, 1, 3).contiguous().to(DEV)
    vd = torch.zeros(n // PS, HD, PS, device=DEV)
    vd[0, :, 0] = 1.0
    T, kv = sum(runs), [n - 37 * (i % 23) for i in range(len(runs))]
    bt = torch.arange(n // PS, dtype=torch.int32, device=DEV).expand(len(runs), -1).contiguous()
    scale = torch.tensor([0.5, 0.75, 1.0, 1.25])[torch.arange(T) % 4]
    q = torch.zeros(T, H, HD)
    for h in range(H):
        q[:, h, h] = scale
    got = torch.empty(T, H * HD, device=DEV)
    K.paged_attention(q.view(T, -1).to(DEV), got, kd.view(-1), vd.view(-1), make_meta(list(zip(runs, kv)), DEV), n_heads=H, n_kv_heads=1, head_dim=HD, page_size=PS, scale=1.0,
                      window=None, block_tables=bt)
    seen = [k - r + i + 1 for r, k in zip(runs, kv) for i in range(r)]
    xd = x[:, :H].double().to(DEV)
    want = torch.stack([1 / torch.exp((xd[:m] - 4.0) * float(c)).sum(0) for m, c in zip(seen, scale)])
    off = (got.view(T, H, HD)[:, :, 5].double() - want) / want
    rms = float(off.pow(2).mean().sqrt()) / EPS
    print(f"rms {rms:.3f} of 2^-24")
    assert rms <= bound


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_attention_float32_values_that_are_not_seen_do_not_count(K, bad):
    """Token 20's value is not a number: queries before it are what they are without it, the ones from it on carry it. A single token whose block
    has no page (a request's page that was given back) gives zeros."""
    from helpers import make_meta
    from test_gpu_kernels import _fill_cache

    H, KVH, HD, PS, runs = 4, 2, 64, 16, [(40, 40), (1, 30)]
    bt, kp, vp, kd, vd, _, _ = _fill_cache(K, torch.float32, [40, 30], KVH, HD, PS, 8, seed=5)
    q = _rand(41, H * HD, seed=6).to(DEV)
    args = dict(n_heads=H, n_kv_heads=KVH, head_dim=HD, page_size=PS, scale=0.125, window=None)
    clean, got = torch.empty(41, H * HD, device=DEV), torch.empty(41, H * HD, device=DEV)
    K.paged_attention(q, clean, kd, vd, make_meta(runs, DEV), block_tables=bt.to(DEV), **args)
    vd.view(-1, KVH, HD, PS)[int(bt[0, 1]), 1, 3, 4] = bad
    bt[1, :] = -1
    K.paged_attention(q, got, kd, vd, make_meta(runs, DEV), block_tables=bt.to(DEV), **args)
    heads = got.view(41, H, HD)
    hit = torch.zeros(41, H, HD, dtype=torch.bool, device=DEV)
    hit[20:40, 2:, 3] = True
    assert bool((~torch.isfinite(heads) == hit).all())
    assert bool((got[40] == 0).all())
    rest = ~hit
    rest[40] = False
    # the other sums of that tile go key by key: another order of at most 40 terms of at most 5, each off by 2^-24 of it
    torch.testing.assert_close(heads[rest], clean.view(41, H, HD)[rest], rtol=0, atol=40 * 5 * EPS)


@pytest.mark.parametrize("HD,H", [(64, 4), (128, 16), (16, 20)])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_attention_float32_values_outside_the_window_do_not_count(K, bad, HD, H):
    """Key 20 holds a value that is not a number, the window 10 keys: of a run and of single tokens only those that see the key carry it."""
    from helpers import make_meta
    from test_gpu_kernels import _fill_cache

    KVH, PS, window, runs = 1, 16, 10, [(40, 40), (1, 30), (1, 31), (1, 21)]
    kv = [k for _, k in runs]
    bt, kp, vp, kd, vd, _, _ = _fill_cache(K, torch.float32, kv, KVH, HD, PS, 12, seed=7)
    T = sum(n for n, _ in runs)
    q = _rand(T, H * HD, seed=8).to(DEV)
    args = dict(n_heads=H, n_kv_heads=KVH, head_dim=HD, page_size=PS, scale=HD ** -0.5, window=window, block_tables=bt.to(DEV))
    clean, got = torch.empty(T, H * HD, device=DEV), torch.empty(T, H * HD, device=DEV)
    K.paged_attention(q, clean, kd, vd, make_meta(runs, DEV), **args)
    for s in range(len(runs)):
        vd.view(-1, KVH, HD, PS)[int(bt[s, 1]), 0, 5, 4] = bad
    K.paged_attention(q, got, kd, vd, make_meta(runs, DEV), **args)
    hit = torch.zeros(T, H, HD, dtype=torch.bool, device=DEV)
    hit[20:30, :, 5] = True  # positions 20 .. 29 see keys 11 .. 29
    hit[[40, 42], :, 5] = True  # positions 29 and 20; position 30 sees 21 .. 30
    heads = got.view(T, H, HD)
    assert bool((~torch.isfinite(heads) == hit).all())
    # the other sums of such a tile go key by key: another order of at most 10 terms of at most 5, each off by 2^-24 of it
    torch.testing.assert_close(heads[~hit], clean.view(T, H, HD)[~hit], rtol=0, atol=10 * 5 * EPS)


# more than 384 workgroups of runs and more than 256 of single tokens (head sizes up to 96): four waves each, of single tokens with a sum for each of a block's two tiles of 16 keys. Key 20 stands in the second tile
# of a window that begins below key 16, in the first of one that begins at 16 to 20, and behind the window of a block's other keys
@pytest.mark.parametrize("HD,H", [(16, 64), (64, 64), (96, 64)])
@pytest.mark.parametrize("window", [10, 60])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_attention_float32_values_outside_the_window_do_not_count_in_four_waves(K, bad, window, HD, H):
    from helpers import make_meta
    from test_gpu_kernels import _fill_cache

    KVH, PS = 16, 16
    kv = [90, *range(18, 35), 79, 80, 81, 100]
    runs = [(90, 90)] + [(1, n) for n in kv[1:]]
    bt, kp, vp, kd, vd, _, _ = _fill_cache(K, torch.float32, kv, KVH, HD, PS, sum(-(-n // PS) for n in kv) + 3, seed=7)
    T = sum(n for n, _ in runs)
    q = _rand(T, H * HD, seed=8).to(DEV)
    args = dict(n_heads=H, n_kv_heads=KVH, head_dim=HD, page_size=PS, scale=HD ** -0.5, window=window, block_tables=bt.to(DEV))
    clean, got = torch.empty(T, H * HD, device=DEV), torch.empty(T, H * HD, device=DEV)
    K.paged_attention(q, clean, kd, vd, make_meta(runs, DEV), **args)
    for s in range(len(runs)):
        vd.view(-1, KVH, HD, PS)[int(bt[s, 1]), :, 5, 4] = bad
    K.paged_attention(q, got, kd, vd, make_meta(runs, DEV), **args)
    pos = torch.tensor([*range(90), *(n - 1 for n in kv[1:])], device=DEV)
    hit = torch.zeros(T, H, HD, dtype=torch.bool, device=DEV)
    hit[(pos >= 20) & (pos < 20 + window), :, 5] = True
    heads = got.view(T, H, HD)
    assert bool((~torch.isfinite(heads) == hit).all())
    # the other sums of such a tile go key by key: another order of at most `window` terms of at most 5, each off by 2^-24 of it
    torch.testing.assert_close(heads[~hit], clean.view(T, H, HD)[~hit], rtol=0, atol=window * 5 * EPS)
