"""head_dim 64 and 96 (bf16 / fp16): probabilities keep fp32's precision in P.V."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from test_gpu_attention import build_case, operator

pytestmark = pytest.mark.gpu

KEYS, HEADS = 5, 16


def one_key_off(device, dtype, d, queries, k_b, factors, values):
    """The last token of five: its score with key 2 is factor * k_b / sqrt(d)
    (one factor per head) and 0 with the others; key i's V is values[i] (per dim,
    dim h being head h's)."""

    q, k, v, cache, md = build_case(device, dtype, [KEYS], [KEYS], HEADS, 1, d, 16, seed=1)
    q.zero_(), k.zero_(), v.zero_()
    q[:, :, 0] = torch.as_tensor(factors, device=device).to(dtype)
    k[2, 0, 0] = k_b
    for i, row in enumerate(values):
        v[i, 0, :HEADS] = torch.as_tensor(row, device=device).to(dtype)
    out = operator()(q, k, v, cache, md)
    if queries == 1:
        last = build_case(device, dtype, [KEYS], [1], HEADS, 1, d, 16, seed=1)[4]
        out = operator()(q[-1:], k[-1:], v[-1:], cache, last)
    return out[-1, :, :HEADS].diagonal().double().cpu().numpy()


def rounded(x):
    return torch.as_tensor(x).float().to(torch.bfloat16).double().numpy()


@pytest.mark.parametrize("d", [64, 96])
@pytest.mark.parametrize("queries", [1, KEYS], ids=["decode", "chunk"])
def test_probabilities_hold_more_than_two_parts_of_bf16(device, d, queries):
    """V takes the first two bf16 parts of a probability p away, so that the
    rest (2.4e-6 .. 3.8e-6 here) is the result, over a sum of 4 + p. The error:
    the score in the exp2 domain is at most 1 with three roundings (1.3e-7 in p),
    the exponential's (1.2e-7), and three sums near 1 (1.2e-7 each at most)."""

    grid = rounded(np.linspace(0.05, 0.69, 4000) * math.sqrt(d))
    p = np.exp(-grid / math.sqrt(d))
    rest = p - rounded(p) - rounded(p - rounded(p))
    chosen = np.unique(grid[np.abs(rest) > 2.4e-6])
    chosen = chosen[np.linspace(0, len(chosen) - 1, HEADS).astype(int)]
    p = np.exp(-chosen / math.sqrt(d))
    hi = rounded(p)
    mid = rounded(p - hi)
    got = one_key_off(device, torch.bfloat16, d, queries, -1.0, chosen, [-hi, -mid, np.ones(HEADS)])
    assert np.abs(got - (p - hi - mid) / (4 + p)).max() < 6.1e-7 / 4


@pytest.mark.parametrize("d", [64, 96])
@pytest.mark.parametrize("queries", [1, KEYS], ids=["decode", "chunk"])
def test_small_probabilities_are_not_rounded_to_fp16_subnormals(device, d, queries):
    """p near 2^-20 lies between fp16's multiples of 2^-24 (up to 3% off). The
    bound: the output's rounding (2^-11) and the score's, 19.6 in the exp2 domain
    with three roundings and the exponential's (1e-5)."""

    grid = torch.linspace(13.0, 14.4, 4000).mul(math.sqrt(d) / 8).half().double().numpy()
    units = np.exp(-8 * grid / math.sqrt(d)) * 2.0**24
    chosen = np.unique(grid[np.abs(units % 1 - 0.5) < 0.2])
    chosen = chosen[np.linspace(0, len(chosen) - 1, HEADS).astype(int)]
    p = np.exp(-8 * chosen / math.sqrt(d))
    zero = np.zeros(HEADS)
    got = one_key_off(device, torch.float16, d, queries, -8.0, chosen, [zero, zero, np.full(HEADS, 30000.0)])
    np.testing.assert_allclose(got, p * 30000.0 / (4 + p), rtol=2.0**-11 + 1e-5)
