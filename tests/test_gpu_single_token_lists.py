"""The list of a step's single tokens in the 32-bit attention and in the one with value heads of their own: any order, behind a run, longer than the step."""
import dataclasses

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("values", [False, True])
def test_any_order_of_single_tokens(values):
    from helpers import make_meta, random_block_tables
    from levanter_amd.kernels import get_kernels

    K, H, G, hd, vd, PS = get_kernels(), 4, 2, 64, 64, 16
    runs = [(3, 40)] + [(1, n) for n in (1, 2, 64, 65, 130, 17, 33)]
    kv, T = [n for _, n in runs], sum(n for n, _ in runs)
    pages = sum(-(-n // PS) for n in kv)
    bt = torch.as_tensor(random_block_tables(kv, PS, pages, 3, "cpu")).to(DEV)
    g = torch.Generator(device=DEV).manual_seed(1)
    dt = torch.bfloat16 if values else torch.float32
    q, k, v = (torch.randn(*s, device=DEV, generator=g).to(dt) for s in ((T, H * hd), (pages, G, hd // 8, PS, 8), (pages, G, vd, PS)))
    outs = []
    in_order = list(range(3, T))
    for order in (in_order, in_order[::-1], in_order[3:] + in_order[:3], in_order * 2):  # the last names every token twice: more entries than the step has tokens
        meta = dataclasses.replace(make_meta(runs, DEV), decode_tokens=torch.tensor(order, dtype=torch.int32, device=DEV), n_decode=len(order))
        out = torch.full((T, H * vd), float("nan"), device=DEV)
        if values:
            K.attention_values(q, out.view(T, H, 1, vd), k, v, meta, n_heads=H, n_kv_heads=G, head_dim=hd, value_dim=vd, all_value_heads=False, page_size=PS, scale=hd ** -0.5,
                               window=None, block_tables=bt)
        else:
            K.paged_attention(q, out, k, v, meta, n_heads=H, n_kv_heads=G, head_dim=hd, page_size=PS, scale=hd ** -0.5, window=None, block_tables=bt)
        outs.append(out)
    assert bool(torch.isfinite(outs[0]).all())
    # the same keys in the same order: the same bits
    for out in outs[1:]:
        assert bool((out == outs[0]).all())
    for t, n in zip(in_order, kv[1:]):
        s = t - 2
        ids = bt[s, :-(-n // PS)].long()
        keys = k[ids].permute(1, 0, 3, 2, 4).reshape(G, -1, hd)[:, :n].double()
        vals = v[ids].permute(1, 0, 3, 2).reshape(G, -1, vd)[:, :n].double()
        for h in range(H):
            p = torch.softmax(keys[h // 2] @ q[t, h * hd:(h + 1) * hd].double() * hd ** -0.5, 0)
            want, size = p @ vals[h // 2], p @ vals[h // 2].abs()
            # bfloat16 weights are off by 2^-9 of them and the scores' rounding; 32-bit ones by the scores' rounding and a few units of the exponential
            assert bool(((outs[0][t, h * vd:(h + 1) * vd].double() - want).abs() <= (2.0 ** -8 if values else 2e-5) * size + 1e-6).all())
