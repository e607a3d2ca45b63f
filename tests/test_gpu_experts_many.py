"""The experts' products over tiles of 128 rows at the edges of the kernel that carries them: outputs that end inside a tile, inner sizes of one step, of an
odd and an even number and with a short step, stretches of one row, of half a tile, a tile and one more or less, output rows without alignment, and lists of
more tiles a chiplet than a wave has lanes."""
import pytest
import torch
import torch.nn.functional as F_

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def K():
    from levanter_amd.kernels import get_kernels

    return get_kernels()


def _sorted(K, counts):
    """One token a pair, in a drawn order; the experts of the sorted pairs beside the lists."""
    E, P = len(counts), sum(counts)
    order = torch.randperm(P, generator=torch.Generator().manual_seed(P))
    chosen = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[order].to(torch.int32).to(DEV).unsqueeze(1)
    tables = torch.empty(2 * P + 1 + 3 * K.moe_max_tiles(P, E, 128), dtype=torch.int32, device=DEV)
    sp, po, meta, tiles = tables[:P], tables[P:2 * P], tables[2 * P:2 * P + 1], tables[2 * P + 1:]
    K.moe_sort(chosen, E, sp, po, tiles, meta, tile_rows=128)
    return sp, tiles, meta, chosen[:, 0].long()[sp.long()]


def _check(K, counts, Fo, Kd, widths, dtypes=(torch.float32, torch.bfloat16)):
    """bfloat16 operands are exact in float64; a sum of Kd products in 32 bits is off by at most Kd * 2^-24 of the sum of their absolute values (e), and
    silu(gate) * up by 1.1 e_gate |up| + |silu(gate)| e_up + 1.1 e_gate e_up (silu's slope stays below 1.1) and 2^-20 of itself."""
    g = torch.Generator(device=DEV).manual_seed(Fo * 31 + Kd)
    E, P = len(counts), sum(counts)
    sp, tiles, meta, expert = _sorted(K, counts)
    h = torch.randn(P, Kd + 8, device=DEV, generator=g).bfloat16()[:, :Kd]
    first = [sum(counts[:e]) for e in range(E)]
    for glu in (False, True):
        w = (torch.randn(E, Fo * (2 if glu else 1), Kd, device=DEV, generator=g) / Kd ** 0.5).bfloat16()
        for gather in (False, True):
            rows = h[sp.long()] if gather else h
            parts = [(rows[first[e]:first[e] + n].double(), w[e].double()) for e, n in enumerate(counts)]
            y = torch.cat([r @ m.T for r, m in parts])
            err = (Kd + 8) * 2.0 ** -24 * torch.cat([r.abs() @ m.abs().T for r, m in parts])
            if glu:
                gate, up, eg, eu = F_.silu(y[:, :Fo]), y[:, Fo:], err[:, :Fo], err[:, Fo:]
                y, err = gate * up, 1.1 * eg * up.abs() + gate.abs() * eu + 1.1 * eg * eu + 2.0 ** -20 * (gate * up).abs()
            for dtype in dtypes:
                for width in widths:
                    out = torch.full((P, width), float("nan"), device=DEV, dtype=dtype)
                    K.moe_linear(h, w, out[:, :Fo], tiles, meta, sp, top=1, gather=gather, glu=glu, activation="silu" if glu else "none", tile_rows=128)
                    bound = err + 1e-30 + (2.0 ** -8 * (y.abs() + err) if dtype is torch.bfloat16 else 0)
                    assert bool(((out[:, :Fo].double() - y).abs() <= bound).all()), (glu, gather, dtype, width)
                    assert bool(torch.isnan(out[:, Fo:]).all())


@pytest.mark.parametrize("Fo", [1, 63, 64, 65, 129])
@pytest.mark.parametrize("Kd", [8, 64, 72, 136, 192, 2056])
def test_products_over_tiles_of_128_rows_against_float64(K, Fo, Kd):
    _check(K, [1, 63, 0, 64, 65, 128, 129], Fo, Kd, (Fo, Fo + 3, (Fo + 3) // 4 * 4 + 4))


@pytest.mark.parametrize("Fo,Kd", [(520, 512), (640, 576), (1032, 1024), (2048, 128)])
def test_columns_that_begin_at_places_of_their_own(K, Fo, Kd):
    """Up to one and a half rounds of workgroups: every column of tiles walks K from another step on; (2048, 128) has more than that with glu."""
    _check(K, [130, 5, 64, 128] if Fo < 2048 else [130, 5, 64, 128] * 6, Fo, Kd, (Fo,))


@pytest.mark.parametrize("activation", ["none", "gelu_new", "gelu", "relu", "silu", "quick_gelu", "tanh", "relu_squared"])
def test_every_activation(K, activation):
    """Against the same sums without one, in float64: an activation's own error is at most 2^-20 of the sum (its slope stays below 1.13; relu_squared's
    is twice the sum), the 32-bit sums are the same in both."""
    f = {"none": lambda x: x, "gelu_new": lambda x: F_.gelu(x, approximate="tanh"), "gelu": F_.gelu, "relu": F_.relu, "silu": F_.silu, "tanh": torch.tanh,
         "quick_gelu": lambda x: x * torch.sigmoid(1.702 * x), "relu_squared": lambda x: F_.relu(x) ** 2}[activation]
    counts, Fo, Kd = [100, 20], 96, 64
    g = torch.Generator(device=DEV).manual_seed(5)
    sp, tiles, meta, _ = _sorted(K, counts)
    h = torch.randn(sum(counts), Kd, device=DEV, generator=g).bfloat16()
    for glu in (False, True):
        w = (torch.randn(2, Fo * (2 if glu else 1), Kd, device=DEV, generator=g) / 6).bfloat16()
        run = lambda w, act, glu: [K.moe_linear(h, w, out := torch.empty(sum(counts), w.shape[1] // (2 if glu else 1), device=DEV), tiles, meta, sp, top=1, gather=False, glu=glu,
                                                activation=act, tile_rows=128), out][1]
        y = run(w, "none", False).double()
        want = f(y[:, :Fo]) * (y[:, Fo:] if glu else 1)
        got = run(w, activation, glu).double()
        bound = 2.0 ** -20 * (1 + y[:, :Fo].abs()) ** 2 * (1 + y[:, Fo:].abs() if glu else 1)
        assert bool(((got - want).abs() <= bound).all())


@pytest.mark.parametrize("experts", [511, 513, 700])
def test_more_tiles_than_lanes_a_chiplet(K, experts):
    """Up to 512 tiles a chiplet's larger ones come first, beyond that the list's order holds."""
    counts = [(1, 130, 200, 70)[e % 4] for e in range(experts - experts // 2)]
    while sum((n + 127) // 128 for n in counts) < experts:
        counts.append(2)
    assert sum((n + 127) // 128 for n in counts) == experts
    _check(K, counts, 72, 136, (72,), (torch.float32,))


@pytest.mark.parametrize("Fo,glu", [(2176, False), (1088, True)])
def test_other_tokens_choices_do_not_change_a_tokens_outputs(K, Fo, glu):
    """The same bits for the tokens of expert 0 beside 31 experts of 128 rows each and beside 16 of 192 and 15 of the rest: 32 and 48 tiles, on either side of
    one and a half rounds of workgroups."""
    E, Kd, P = 32, 512, 4096
    g = torch.Generator(device=DEV).manual_seed(3)
    h = torch.randn(P, Kd, device=DEV, generator=g).bfloat16()
    w = (torch.randn(E, Fo * (2 if glu else 1), Kd, device=DEV, generator=g) / Kd ** 0.5).bfloat16()
    outs = []
    for counts in ([128] * 32, [128] + [192] * 16 + [60] * 11 + [59] * 4):
        chosen = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).to(torch.int32).to(DEV).unsqueeze(1)
        tables = torch.empty(2 * P + 1 + 3 * K.moe_max_tiles(P, E, 128), dtype=torch.int32, device=DEV)
        sp, po, meta, tiles = tables[:P], tables[P:2 * P], tables[2 * P:2 * P + 1], tables[2 * P + 1:]
        K.moe_sort(chosen, E, sp, po, tiles, meta, tile_rows=128)
        out = torch.empty(P, Fo, device=DEV)
        K.moe_linear(h, w, out, tiles, meta, sp, top=1, gather=True, glu=glu, activation="silu" if glu else "none", tile_rows=128)
        outs.append(out[po.long()][:128])
    assert torch.equal(*outs)
