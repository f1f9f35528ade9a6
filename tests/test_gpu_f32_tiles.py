"""fp32 attention on the fp32 matrix cores against the oracle and against the
any-shape kernel (which a query that is not 16-byte aligned still takes)."""

from __future__ import annotations

import dataclasses

import pytest
import torch

from micro_vllm_amd.attention import ChunkedLocalSpec, SlidingWindowSpec
from test_gpu_attention import build_case, operator, run_and_check

pytestmark = pytest.mark.gpu

LENGTHS = [1, 15, 16, 17, 2, 17, 127, 128, 129, 700, 1500, 5]
QLENS = [1, 1, 1, 1, 2, 17, 1, 9, 129, 33, 1, 5]


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize(("hq", "hkv"), [(4, 4), (16, 8), (14, 2), (32, 2), (9, 3), (17, 1)], ids=str)
@pytest.mark.parametrize(("bs", "spec"), [(16, None), (5, SlidingWindowSpec(100)), (48, ChunkedLocalSpec(48))], ids=str)
def test_groups_tiles_and_specs(device, d, hq, hkv, bs, spec):
    """Groups that leave columns of the 16 empty (7, 9 and, beyond the kernel,
    17), chunks that end inside a token block, tiles cut by windows."""

    q, k, v, cache, md = build_case(device, torch.float32, LENGTHS, QLENS, hq, hkv, d, bs, spec=spec, seed=hq + d)
    run_and_check(q, k, v, cache, md, torch.float32)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize(("hq", "hkv"), [(16, 8), (16, 1)], ids=str)
def test_long_contexts(device, d, hq, hkv):
    """Contexts of many rounds of the eight waves' tiles, one of them a chunk."""

    q, k, v, cache, md = build_case(device, torch.float32, [20_000, 8193, 9001], [1, 1, 7], hq, hkv, d, 16, seed=d)
    run_and_check(q, k, v, cache, md, torch.float32)


@pytest.mark.parametrize("requests", [1, 63, 64, 65, 700, 4100])
def test_request_search(device, requests):
    """The 64-ary search over one, two and three rounds, empty requests between."""

    lengths = [1 + (r * 7) % 40 for r in range(requests)]
    qlens = [min(n, 1 + r % 3) for r, n in enumerate(lengths)]
    q, k, v, cache, md = build_case(device, torch.float32, lengths, qlens, 2, 1, 64, 16, seed=requests)
    run_and_check(q, k, v, cache, md, torch.float32)


def shifted(q):
    out = torch.empty(q.numel() + 1, dtype=q.dtype, device=q.device)[1:].view(q.shape)
    out.copy_(q)
    assert out.data_ptr() % 16 != 0
    return out


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_values_that_are_not_finite_reach_only_rows_that_see_them(device, bad):
    """Tokens of one block share V tiles; a later token's non-finite V row
    stays out of the earlier tokens, as in the any-shape kernel. Peaked scores
    rescale the accumulators. The bound: q.k has 128 terms of rms 6 and partial
    sums up to ~200, so its rounding (sqrt(128) errors of 2^-25 * 200) over
    sqrt(128) is ~6e-6 at most in a score, hence in p; times |v| up to 4, 2.4e-5."""

    q, k, v, cache, md = build_case(device, torch.float32, LENGTHS, QLENS, 16, 8, 128, 16, seed=3)
    q = q * 6
    v[40, 3, 5] = bad
    v[100, 1, 77] = bad
    expected = operator()(shifted(q), k, v, cache.clone(), md)
    got = operator()(q, k, v, cache, md)
    assert not torch.isfinite(expected).all() and torch.isfinite(expected[:20]).all()
    torch.testing.assert_close(got, expected, rtol=2e-5, atol=2.4e-5, equal_nan=True)


def test_rows_outside_every_request_and_without_keys(device):
    q, k, v, cache, md = build_case(device, torch.float32, [50, 40, 30], [3, 1, 2], 16, 8, 128, 16, seed=2)
    pad = lambda t, value: torch.cat([t, torch.full((70, *t.shape[1:]), value, dtype=t.dtype, device=device)])  # noqa: E731
    starts = md.query_context_start_positions.clone()
    starts[3] = md.query_positions[3] + 1  # the single-token request sees nothing
    md = dataclasses.replace(
        md, query_positions=pad(md.query_positions, 0), query_context_start_positions=pad(starts, 0),
        slot_mapping=pad(md.slot_mapping, -1),
    )
    q, k, v = pad(q, 1.0), pad(k, 1.0), pad(v, 1.0)
    expected = operator()(shifted(q), k, v, cache.clone(), md)
    got = operator()(q, k, v, cache, md)
    assert torch.isnan(got[3]).all() and (got[6:] == 0).all()
    torch.testing.assert_close(got, expected, rtol=2e-5, atol=2e-6, equal_nan=True)
