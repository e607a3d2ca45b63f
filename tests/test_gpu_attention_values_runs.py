"""Runs of several tokens in the attention with value heads of their own, where its workgroups end: against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PS = 16


def _step(runs):
    """(new tokens, keys) a run -> the step's description, block tables, number of pages; page ids are dealt from the last on."""
    from levanter_amd.kernels import get_kernels
    from levanter_amd.parts.base import AttentionMeta

    rows = get_kernels().prefill_tile_rows
    pos, seq, tiles, t = [], [], [], 0
    for i, (n, kv) in enumerate(runs):
        pos += range(kv - n, kv)
        seq += [i] * n
        tiles += [(t + r, min(rows, n - r)) for r in range(0, n, rows)]
        t += n
    need = [-(-kv // PS) for _, kv in runs]
    bt, last = torch.full((len(runs), max(need) + 1), -1, dtype=torch.int32), sum(need)
    for i, k in enumerate(need):
        bt[i, :k] = torch.arange(last - 1, last - 1 - k, -1)
        last -= k
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    return AttentionMeta(ints(pos), ints(seq), ints(tiles), len(tiles), None, 0, max(kv for _, kv in runs)), bt.to(DEV), sum(need)


# workgroups of 64 query tokens (keys and values of a head up to 192 numbers together) and of 128; key and value sizes that are no multiple of 32 and of two tiles; every
# key/value head's values, too. Run lengths end one before, at and behind a workgroup's and a block of keys' last token; windows begin inside a block.
@pytest.mark.parametrize("dk,dv,H,G,all_values", [(128, 64, 4, 2, False), (16, 16, 2, 1, False), (48, 32, 2, 2, False), (144, 112, 2, 1, False), (256, 224, 2, 1, False), (64, 48, 4, 2, False),
                                                  (128, 64, 4, 4, True), (48, 32, 4, 2, True), (64, 48, 2, 2, True)])
@pytest.mark.parametrize("window,softcap", [(None, None), (70, None), (None, 4.0)])
def test_runs(dk, dv, H, G, all_values, window, softcap):
    _check([(63, 63), (64, 64), (65, 129), (127, 140), (128, 128), (129, 193), (2, 300), (200, 391)], dk, dv, H, G, all_values, window, softcap)


# half empty tiles, contexts of up to 256 keys and longer ones, and more tiles than half tiles would be on the chip at once (400 and 448 of a tile and a head): whole tiles a workgroup
@pytest.mark.parametrize("dk,dv,H,G", [(128, 64, 4, 2), (16, 16, 2, 1), (48, 32, 2, 2), (144, 112, 2, 1), (256, 224, 2, 1), (128, 128, 2, 1)])
@pytest.mark.parametrize("runs,many", [([(2, 2), (63, 63), (64, 64), (65, 129), (17, 256), (16, 80)], 1), ([(31, 300), (64, 391), (2, 65)], 1), ([(128, 128), (66, 66), (127, 140), (129, 193), (100, 391)], 32)])
def test_runs_in_whole_tiles(dk, dv, H, G, runs, many):
    _check(runs, dk, dv, H * many, G, False, 70, None)


def _check(runs, dk, dv, H, G, all_values, window, softcap):
    from levanter_amd.kernels import get_kernels

    meta, bt, pages = _step(runs)
    g = torch.Generator(device=DEV).manual_seed(dk + dv)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    T = sum(n for n, _ in runs)
    q, k, v = rnd(T, H * dk).bfloat16(), rnd(pages, G, dk // 8, PS, 8).bfloat16(), rnd(pages, G, dv, PS).bfloat16()
    slopes, sinks = torch.rand(H, device=DEV, generator=g) * 0.02, rnd(H)
    for i, (_, kv) in enumerate(runs):  # behind a run's last key a page may hold anything
        page, at = int(bt[i, (kv - 1) // PS]), (kv - 1) % PS + 1
        k[page, :, :, at:], v[page, :, :, at:] = float("nan"), float("nan")
    nv = G if all_values else 1
    out = torch.full((T, H, nv, dv), float("nan"), device=DEV)
    get_kernels().attention_values(q, out, k, v, meta, n_heads=H, n_kv_heads=G, head_dim=dk, value_dim=dv, all_value_heads=all_values, page_size=PS, scale=dk ** -0.5,
                                   window=window, block_tables=bt, softcap=softcap, slopes=slopes, sinks=sinks)
    t = 0
    for i, (n, kv) in enumerate(runs):
        ids = bt[i, :-(-kv // PS)].long()
        K = k[ids].permute(1, 0, 3, 2, 4).reshape(G, -1, dk)[:, :kv].double()
        V = v[ids].permute(1, 0, 3, 2).reshape(G, -1, dv)[:, :kv].double()
        far = (torch.arange(kv - n, kv, device=DEV)[:, None] - torch.arange(kv, device=DEV)[None]).double()
        Q = q[t:t + n].view(n, H, dk).permute(1, 0, 2).double()
        s = torch.stack([Q[h] @ K[h * G // H].T for h in range(H)]) * dk ** -0.5
        s = softcap * torch.tanh(s / softcap) if softcap else s
        s = s - slopes.double()[:, None, None] * far
        s = s.masked_fill((far < 0) | (far >= (window or kv)), -float("inf"))
        p = torch.softmax(torch.cat([s, sinks.double()[:, None, None].expand(H, n, 1)], 2), 2)[:, :, :kv]
        for h in range(H):
            for c in range(nv):
                head = c if all_values else h * G // H
                want, size = p[h] @ V[head], p[h] @ V[head].abs()
                # a weight is rounded to bfloat16 (2^-9 of it), scores and their exponentials in 32 bits with the hardware's functions: 2^-8 covers both
                assert bool(((out[t:t + n, h, c].double() - want).abs() <= 2.0 ** -8 * size + 1e-6).all())
        t += n
