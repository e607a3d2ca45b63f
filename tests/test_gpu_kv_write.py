"""New keys and values into their pages: portions that begin and end anywhere in a page, tokens that are dropped, single tokens between portions, rows
without alignment, heads of one chunk and heads whose values have another size. Copies: every byte is compared, also those no token goes to."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("KVH,HD,VD,PS", [(1, 8, 8, 16), (3, 64, 64, 16), (2, 128, 96, 48), (2, 24, 200, 32)])
@pytest.mark.parametrize("aligned", [True, False])
def test_tokens_into_shuffled_pages(dtype, KVH, HD, VD, PS, aligned):
    from levanter_amd.kernels import get_kernels

    g = torch.Generator().manual_seed(HD + VD + PS)
    dest, page, n_pages = [], 0, 64
    order = torch.randperm(n_pages, generator=g).tolist()
    for start, n in ((0, 16), (3, 29), (8, 8), (5, 1), (15, 1), (7, 40), (0, 1), (9, 17)):  # each in pages of its own
        dest += [order[page + (start + i) // PS] * PS + (start + i) % PS for i in range(n)]
        page += (start + n - 1) // PS + 1
    for at in (1, 20, 50, len(dest) - 1):
        dest[at] = -1
    T, pad = len(dest), 8 if aligned else 1
    k = torch.randn(T, KVH * HD + pad, generator=g).to(dtype).to(DEV)[:, :KVH * HD]
    v = torch.randn(T, KVH * VD + pad, generator=g).to(dtype).to(DEV)[:, :KVH * VD]
    kp = torch.full((n_pages, KVH, HD // 8, PS, 8), float("nan"), dtype=dtype, device=DEV)
    vp = torch.full((n_pages, KVH, VD, PS), float("nan"), dtype=dtype, device=DEV)
    want_k, want_v = kp.cpu(), vp.cpu()
    for t, d in enumerate(dest):
        if d >= 0:
            want_k[d // PS, :, :, d % PS] = k[t].cpu().view(KVH, HD // 8, 8)
            want_v[d // PS, :, :, d % PS] = v[t].cpu().view(KVH, VD)
    get_kernels().kv_write(k, v, kp, vp, torch.tensor(dest, dtype=torch.int32, device=DEV), KVH, HD, PS, VD)
    assert torch.equal(kp.cpu().nan_to_num(7.0), want_k.nan_to_num(7.0)) and torch.equal(vp.cpu().nan_to_num(7.0), want_v.nan_to_num(7.0))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("KVH,HD,VD", [(3, 64, 64), (2, 128, 96), (1, 8, 8)])
@pytest.mark.parametrize("singles", [1, 7, 9, 10, 11, 15, 16, 37])
def test_single_tokens_ahead_of_a_portion(dtype, KVH, HD, VD, singles):
    """Single tokens anywhere in pages of their own, some dropped, then a portion that begins inside a workgroup's tokens at any slot of a page."""
    from levanter_amd.kernels import get_kernels

    PS, g = 16, torch.Generator().manual_seed(singles)
    slots = torch.randint(0, PS, (singles,), generator=g).tolist()
    for start in (0, 3, 8, 13):
        n_pages = singles + 5
        order = torch.randperm(n_pages, generator=g).tolist()
        dest = [order[i] * PS + s if i % 6 != 5 else -1 for i, s in enumerate(slots)] + [order[singles + (start + i) // PS] * PS + (start + i) % PS for i in range(50)]
        T = len(dest)
        k, v = (torch.randn(T, KVH * d, generator=g).to(dtype).to(DEV) for d in (HD, VD))
        kp = torch.full((n_pages, KVH, HD // 8, PS, 8), float("nan"), dtype=dtype, device=DEV)
        vp = torch.full((n_pages, KVH, VD, PS), float("nan"), dtype=dtype, device=DEV)
        want_k, want_v = kp.cpu(), vp.cpu()
        for t, d in enumerate(dest):
            if d >= 0:
                want_k[d // PS, :, :, d % PS] = k[t].cpu().view(KVH, HD // 8, 8)
                want_v[d // PS, :, :, d % PS] = v[t].cpu().view(KVH, VD)
        get_kernels().kv_write(k, v, kp, vp, torch.tensor(dest, dtype=torch.int32, device=DEV), KVH, HD, PS, VD)
        assert torch.equal(kp.cpu().nan_to_num(7.0), want_k.nan_to_num(7.0)) and torch.equal(vp.cpu().nan_to_num(7.0), want_v.nan_to_num(7.0))
