"""Attention whose weights go to every value head: numbers of value heads at and beside what a wave has room for (one, two, four, eight), single tokens whose
keys are one block, several, and split over waves, beside short runs; against float64."""
import math

import pytest
import torch

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
