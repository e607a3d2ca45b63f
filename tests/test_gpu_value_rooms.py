"""Attention whose weights go to every value head: numbers of value heads at and beside what a wave has room for (one, two, four, eight), single tokens whose
keys are one block, several, and split over waves, beside short runs; against float64."""
import math

import pytest
import torch

from helpers import make_meta, random_block_tables
from test_gpu_zederax import Z, as_bf16_numbers, plain_attention, run_attention, tol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,dk,dv", [(1, 32, 32), (2, 32, 32), (3, 32, 32), (5, 32, 32), (8, 32, 32), (9, 32, 32), (1, 64, 64), (2, 64, 64), (4, 64, 64), (7, 64, 64),
                                     (1, 128, 128), (2, 128, 128), (3, 128, 128)])
@pytest.mark.parametrize("talking", [True, False])
def test_every_number_of_value_heads(G, dk, dv, talking):
    """The tolerance is that of the attention tests beside it: weights and values in bfloat16."""
    H = 2 * G
    g = torch.Generator().manual_seed(G * 100 + dk)
    runs = [(1, 1), (1, 63), (1, 64), (1, 65), (1, 300), (1, 1030), (3, 70), (17, 17)]
    q, k = ([as_bf16_numbers(Z.unit_rms(torch.randn(r[i], n, dk, generator=g), 1e-6).reshape(r[i], -1)) for r in runs] for i, n in ((0, H), (1, G)))
    v = [as_bf16_numbers(torch.randn(kl, G * dv, generator=g)) for _, kl in runs]
    T = sum(ql for ql, _ in runs)
    talk = as_bf16_numbers(torch.eye(H) + 0.5 * torch.randn(H, H, generator=g)) if talking else None
    gate = as_bf16_numbers(torch.randn(T, H, generator=g)) if talking else None
    args = (H, G, dk, dv, runs, 200, 20.0, 4.0 / math.sqrt(dk), q, k, v, talk, gate)
    torch.testing.assert_close(run_attention(torch.bfloat16, *args), plain_attention(*args), **tol(torch.bfloat16, bf16=3e-2))


@pytest.mark.parametrize("ps", [16, 48, 64, 80, 128])
@pytest.mark.parametrize("G,dk,dv,talking", [(2, 128, 64, False), (2, 64, 32, True)])
@pytest.mark.parametrize("window", [None, 70, 64])
def test_page_sizes_of_runs(ps, G, dk, dv, talking, window):
    """Runs that begin and end beside the blocks of 64 keys and beside pages of several sizes, as against the float64 statement."""
    H = 2 * G
    g = torch.Generator().manual_seed(ps * 10 + dk)
    runs = [(128, 128), (129, 129), (130, 261), (64, 127), (257, 700), (2, 65)]
    q, k = ([as_bf16_numbers(Z.unit_rms(torch.randn(r[i], n, dk, generator=g), 1e-6).reshape(r[i], -1)) for r in runs] for i, n in ((0, H), (1, G)))
    v = [as_bf16_numbers(torch.randn(kl, G * dv, generator=g)) for _, kl in runs]
    talk = as_bf16_numbers(torch.eye(H) + 0.5 * torch.randn(H, H, generator=g)) if talking else None
    args = (H, G, dk, dv, runs, window, None, 4.0 / math.sqrt(dk), q, k, v, talk, None)
    torch.testing.assert_close(run_attention(torch.bfloat16, *args, ps=ps), plain_attention(*args), **tol(torch.bfloat16, bf16=3e-2))


@pytest.mark.parametrize("ps,window,keep", [(16, 70, 0), (16, 100, 5), (48, 70, 33), (64, 130, 70), (128, 64, 0)])
def test_pages_out_of_sight_are_not_there(ps, window, keep):
    """A run's pages that hold no key in sight are given back (-1 in the table), what they held and what a recycled page holds is NaN: the same bits as with
    all pages there."""
    from levanter_amd.kernels import get_kernels

    kern, H, G, dk, dv = get_kernels(), 4, 2, 128, 64
    runs, dev = [(130, 515), (70, 300)], "cuda:0"
    g = torch.Generator(device=dev).manual_seed(ps + window)
    lens = [n for _, n in runs]
    pages = sum(-(-n // ps) for n in lens)
    bt = random_block_tables(lens, ps, pages + 1, 1, dev)
    q = torch.randn(sum(n for n, _ in runs), H * dk, device=dev, generator=g).bfloat16()
    k_pages, v_pages = (torch.randn(pages + 1, G * d * ps, device=dev, generator=g).bfloat16() for d in (dk, dv))
    outs = []
    for released in (False, True):
        if released:
            for r, (ql, kl) in enumerate(runs):
                for b in range(-(-kl // ps)):
                    if (b + 1) * ps <= kl - ql - window + 1 and b * ps >= keep:
                        k_pages[bt[r, b]] = float("nan")
                        v_pages[bt[r, b]] = float("nan")
                        bt[r, b] = -1
            assert bool((bt[:, :-(-min(lens) // ps)] < 0).any())
        out = torch.empty(q.shape[0], H, 1, dv, device=dev)
        kern.attention_values(q, out, k_pages, v_pages, make_meta(runs, dev), n_heads=H, n_kv_heads=G, head_dim=dk, value_dim=dv, all_value_heads=False, page_size=ps,
                              scale=dk ** -0.5, window=window, block_tables=bt, keep_first=keep)
        outs.append(out)
    assert bool(torch.isfinite(outs[0]).all()) and torch.equal(*outs)


@pytest.mark.parametrize("G,dk,dv,talking", [(1, 128, 64, False), (2, 64, 32, True), (1, 256, 224, False), (3, 32, 32, True)])
@pytest.mark.parametrize("keys", [65, 128, 129, 250, 257, 449, 512, 513])
@pytest.mark.parametrize("window", [None, 100])
def test_ranges_of_keys_that_one_workgroup_merges(G, dk, dv, talking, keys, window):
    """Two to nine ranges of a single token's keys, beside tokens with fewer keys than there are ranges: up to four or eight are merged by the waves of a
    workgroup, more by a kernel of their own."""
    H = 2 * G
    g = torch.Generator().manual_seed(keys + dk)
    runs = [(1, keys), (1, 1), (1, 64), (1, max(1, keys - 1))]
    q, k = ([as_bf16_numbers(Z.unit_rms(torch.randn(r[i], n, dk, generator=g), 1e-6).reshape(r[i], -1)) for r in runs] for i, n in ((0, H), (1, G)))
    v = [as_bf16_numbers(torch.randn(kl, G * dv, generator=g)) for _, kl in runs]
    talk = as_bf16_numbers(torch.eye(H) + 0.5 * torch.randn(H, H, generator=g)) if talking else None
    args = (H, G, dk, dv, runs, window, None, 4.0 / math.sqrt(dk), q, k, v, talk, None)
    torch.testing.assert_close(run_attention(torch.bfloat16, *args), plain_attention(*args), **tol(torch.bfloat16, bf16=3e-2))


@pytest.mark.parametrize("G,dk,dv,talking", [(1, 128, 64, False), (2, 64, 32, True), (1, 256, 224, False), (3, 32, 32, True)])
@pytest.mark.parametrize("keys", [65, 129, 250, 449])
def test_a_workgroups_merge_is_the_second_kernels(G, dk, dv, talking, keys):
    """The same ranges, merged by their workgroup without scratch memory and, the step said to reach so many keys that its reads would crowd a CU, by the
    second kernel: the same bits."""
    from levanter_amd.kernels import build, get_kernels

    kern, H, ps, dev = get_kernels(), 2 * G, 16, "cuda:0"
    lens = [keys, 1, 64, keys - 1]
    g = torch.Generator(device=dev).manual_seed(keys + dk)
    pages = sum(-(-n // ps) for n in lens)
    bt = random_block_tables(lens, ps, pages, 1, dev)
    q = torch.randn(len(lens), H * dk, device=dev, generator=g).bfloat16()
    k_pages, v_pages = (torch.randn(pages, G * d * ps, device=dev, generator=g).bfloat16() for d in (dk, dv))
    nv = G if talking else 1
    sinks = torch.randn(H, device=dev, generator=g)
    meta, outs = make_meta([(1, n) for n in lens], dev), []
    lib = kern._unit(build.attention_values_unit(dk, dv))
    for many in (False, True):
        if many:
            ((key, (splits, scratch)),) = meta.plans.items()
            if splits == 1 or (splits > 4 and dk == 256):
                return  # one range, or more than a workgroup merges
            assert scratch is None
            meta.max_kv_len = 1 << 20
            need = lib.lev_attention_values_mfma_workspace(len(lens), splits, H, G, nv, 0, 0, 0, meta.max_kv_len)
            assert need == len(lens) * splits * H * (nv * dv + 2) * 4
            meta.plans[key] = (splits, torch.empty(need, dtype=torch.uint8, device=dev))
        out = torch.empty(len(lens), H, nv, dv, device=dev)
        kern.attention_values(q, out, k_pages, v_pages, meta, n_heads=H, n_kv_heads=G, head_dim=dk, value_dim=dv, all_value_heads=talking, page_size=ps,
                              scale=dk ** -0.5, window=None, block_tables=bt, sinks=sinks)
        outs.append(out)
    assert torch.equal(*outs)
