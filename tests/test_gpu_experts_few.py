"""The experts' products over tiles of 16 rows at the edges of the kernel that carries them: outputs that end inside a tile, inner sizes with a short
last chunk and with fewer pairs of k-steps than waves, both numbers of waves, stretches of one row, of a tile and of one more, output rows without alignment."""
import pytest
import torch
import torch.nn.functional as F_

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def K():
    from levanter_amd.kernels import get_kernels

    return get_kernels()


@pytest.mark.parametrize("F", [1, 8, 15, 16, 17, 100])
@pytest.mark.parametrize("Kd", [8, 64, 72, 520, 2040, 2048, 2056, 3080])
def test_products_over_tiles_of_16_rows_against_float64(K, F, Kd):
    """bfloat16 operands are exact in float64; a sum of Kd products in 32 bits is off by at most Kd * 2^-24 of the sum of their absolute values (e), and
    silu(gate) * up by 1.1 e_gate |up| + |silu(gate)| e_up + 1.1 e_gate e_up (silu's slope stays below 1.1) and 2^-20 of itself."""
    g = torch.Generator(device=DEV).manual_seed(F * 31 + Kd)
    counts = [1, 0, 16, 17, 40, 3]  # rows of each expert; one token a pair
    E, P = len(counts), sum(counts)
    chosen = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(P)].to(torch.int32).to(DEV).unsqueeze(1)
    h = torch.randn(P, Kd + 8, device=DEV, generator=g).bfloat16()[:, :Kd]
    tables = torch.empty(2 * P + 1 + 3 * K.moe_max_tiles(P, E, 16), dtype=torch.int32, device=DEV)
    sp, po, meta, tiles = tables[:P], tables[P:2 * P], tables[2 * P:2 * P + 1], tables[2 * P + 1:]
    K.moe_sort(chosen, E, sp, po, tiles, meta, tile_rows=16)
    expert = chosen[:, 0].long()[sp.long()]
    for glu in (False, True):
        w = (torch.randn(E, F * (2 if glu else 1), Kd, device=DEV, generator=g) / Kd ** 0.5).bfloat16()
        for gather in (False, True):
            rows = (h[sp.long()] if gather else h).double()
            y = torch.stack([w[e].double() @ r for e, r in zip(expert.tolist(), rows)])
            err = (Kd + 8) * 2.0 ** -24 * torch.stack([w[e].double().abs() @ r.abs() for e, r in zip(expert.tolist(), rows)])
            if glu:
                gate, up, eg, eu = F_.silu(y[:, :F]), y[:, F:], err[:, :F], err[:, F:]
                y, err = gate * up, 1.1 * eg * up.abs() + gate.abs() * eu + 1.1 * eg * eu + 2.0 ** -20 * (gate * up).abs()
            for dtype in (torch.float32, torch.bfloat16):
                for width in (F, F + 3, (F + 3) // 4 * 4 + 4):
                    out = torch.full((P, width), float("nan"), device=DEV, dtype=dtype)
                    K.moe_linear(h, w, out[:, :F], tiles, meta, sp, top=1, gather=gather, glu=glu, activation="silu" if glu else "none", tile_rows=16)
                    bound = err + 1e-30 + (2.0 ** -8 * (y.abs() + err) if dtype is torch.bfloat16 else 0)
                    assert bool(((out[:, :F].double() - y).abs() <= bound).all()), (glu, gather, dtype, width)
                    assert bool(torch.isnan(out[:, F:]).all())


@pytest.mark.parametrize("Kd,sums", [(1024, 8), (2048, 16)])
def test_the_sums_chains_of_roundings_stay_short(K, Kd, sums):
    """The error in root mean square of Kd products in ``sums`` partial sums, derived as in the test of the same name in test_gpu_skinny.py."""
    g = torch.Generator(device=DEV).manual_seed(Kd)
    T, E, F = 8, 4, 1024
    chosen = (torch.arange(T) % E).to(torch.int32).to(DEV).unsqueeze(1)
    h, w = torch.randn(T, Kd, device=DEV, generator=g).bfloat16(), torch.randn(E, F, Kd, device=DEV, generator=g).bfloat16()
    tables = torch.empty(2 * T + 1 + 3 * K.moe_max_tiles(T, E, 16), dtype=torch.int32, device=DEV)
    sp, po, meta, tiles = tables[:T], tables[T:2 * T], tables[2 * T:2 * T + 1], tables[2 * T + 1:]
    K.moe_sort(chosen, E, sp, po, tiles, meta, tile_rows=16)
    out = torch.empty(T, F, device=DEV)
    K.moe_linear(h, w, out, tiles, meta, sp, top=1, gather=True, tile_rows=16)
    want = torch.stack([w[t % E].double() @ h[t].double() for t in sp.tolist()])
    error, n = float((out.double() - want).norm() / want.norm()), Kd / 32 / sums
    assert error <= 1.06 * 0.40 * 2.0 ** -24 * ((4 * n + 1) / 2 + (sums + 1) / 2) ** 0.5, error
