"""32-bit attention of single tokens that writes the step's keys and values itself: the same output as writing them first, and the same pages, bit for bit."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def K():
    from levanter_amd.kernels import get_kernels

    return get_kernels()


@pytest.mark.parametrize("H,KVH,HD,PS,lens,window,odd", [
    (12, 12, 64, 16, [1, 16, 17, 203, 257], None, False), (16, 4, 96, 32, [33, 512, 100], None, False), (40, 1, 128, 16, [40, 300], None, False),  # 40 heads of one: three workgroups
    (3, 3, 16, 16, [1, 2, 700], 64, False), (12, 12, 64, 16, [5, 96, 255], None, True)])
def test_written_on_the_way(K, H, KVH, HD, PS, lens, window, odd):
    from test_gpu_kernels import _fill_cache, make_meta

    n_pages = sum((n + PS - 1) // PS for n in lens) + 2
    bt, _, _, k1, v1, _, _ = _fill_cache(K, torch.float32, lens, KVH, HD, PS, n_pages, seed=3)
    k2, v2 = k1.clone(), v1.clone()
    g = torch.Generator(device=DEV).manual_seed(1)
    T, D = len(lens), KVH * HD
    qkv = torch.randn(T, H * HD + 2 * D, device=DEV, generator=g)
    q, k, v = qkv[:, :H * HD], qkv[:, H * HD:H * HD + D], qkv[:, H * HD + D:]
    if odd:  # a new value that is not finite takes the path that goes key by key
        v[1, 3] = float("inf")
    dest = torch.tensor([int(bt[i, (n - 1) // PS]) * PS + (n - 1) % PS for i, n in enumerate(lens)], dtype=torch.int32, device=DEV)
    meta = make_meta([(1, n) for n in lens], DEV)
    args = dict(n_heads=H, n_kv_heads=KVH, head_dim=HD, page_size=PS, scale=1 / math.sqrt(HD), window=window, block_tables=bt.to(DEV))
    out1, out2 = (torch.full((T, H * HD), float("nan"), device=DEV) for _ in range(2))
    nan = torch.full((T, D), float("nan"), device=DEV)
    K.kv_write(nan, nan, k2, v2, dest, KVH, HD, PS)
    K.kv_write(k, v, k1, v1, dest, KVH, HD, PS)
    assert K.paged_attention(q, out1, k1, v1, meta, **args) is False
    assert K.paged_attention(q, out2, k2, v2, meta, k_new=k, v_new=v, dest=dest, **args) is True
    torch.testing.assert_close(out2, out1, rtol=0, atol=0, equal_nan=True)
    assert torch.equal(k1.view(torch.int32), k2.view(torch.int32)) and torch.equal(v1.view(torch.int32), v2.view(torch.int32))


@pytest.mark.parametrize("odd", [False, True])
def test_written_on_the_way_by_four_waves(K, odd):
    """More than 256 workgroups have four waves each: the one behind the last keys' wave is the writer, also where that is the first again."""
    test_written_on_the_way(K, 16, 16, 64, 16, [1, 5, 31, 32, 33, 64, 65, 96, 97, 127, 128, 129, 160, 161, 255, 256, 300], None, odd)
