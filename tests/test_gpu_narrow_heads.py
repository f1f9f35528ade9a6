"""head_dim 64 and 96 (bf16 / fp16) on the matrix-core kernels.

Checked against the oracle at the sizes where tiles end (16-token decode
tiles, 64-key prefill tiles, 128-row workgroups, split boundaries), and
against the any-shape kernel, which a query view that is not 16-byte aligned
still takes.
"""

from __future__ import annotations

import pytest
import torch

from micro_vllm_amd.attention import ChunkedLocalSpec, SlidingWindowSpec
from micro_vllm_amd.attention.operators.mi355x_paged import AttentionPlan, hip_attention_over_cache
from test_gpu_attention import build_case, operator, run_and_check

pytestmark = pytest.mark.gpu

LENGTHS = [1, 15, 16, 17, 64, 65, 700, 2, 17, 129, 600, 90, 1100, 3000]
QLENS = [1, 1, 1, 1, 1, 1, 1, 2, 17, 100, 600, 3, 33, 1]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 96])
@pytest.mark.parametrize(("hq", "hkv"), [(8, 8), (32, 8), (14, 2), (16, 1), (6, 3)], ids=str)
def test_group_sizes_and_tile_edges(device, dtype, d, hq, hkv):
    """Groups of 7 take the decode kernel beside the any-shape kernel's
    chunks; one and three KV heads leave waves of a workgroup without one."""

    q, k, v, cache, md = build_case(device, dtype, LENGTHS, QLENS, hq, hkv, d, 16, seed=d + hq)
    run_and_check(q, k, v, cache, md, dtype)


@pytest.mark.parametrize("d", [64, 96])
@pytest.mark.parametrize("bs", [8, 32, 48, 256])
@pytest.mark.parametrize("spec", [None, SlidingWindowSpec(1), SlidingWindowSpec(100), ChunkedLocalSpec(48)], ids=repr)
def test_block_sizes_and_bounded_specs(device, d, bs, spec):
    q, k, v, cache, md = build_case(device, torch.bfloat16, LENGTHS, QLENS, 8, 2, d, bs, spec=spec, seed=d + bs)
    run_and_check(q, k, v, cache, md, torch.bfloat16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 96])
@pytest.mark.parametrize("scale", [1.0, 12.0], ids=["flat", "peaked"])
def test_agrees_with_the_any_shape_kernel(device, dtype, d, scale):
    """Both hold the probabilities to at least 16 bits of mantissa and round
    once, so results differ by one unit in the last place at most, plus
    2^-17 of the largest |v| (about 4) where they nearly cancel; also with
    scores that jump by many powers of two (rescaled accumulators)."""

    q, k, v, cache, md = build_case(device, dtype, LENGTHS, QLENS, 16, 4, d, 16, seed=5)
    q = q * scale
    shifted = torch.empty(q.numel() + 1, dtype=dtype, device=device)[1:].view(q.shape)
    shifted.copy_(q)
    assert shifted.data_ptr() % 16 != 0
    general = operator()(shifted, k, v, cache.clone(), md)
    got = operator()(q, k, v, cache, md)
    ulp = 2.0**-7 if dtype == torch.bfloat16 else 2.0**-10
    torch.testing.assert_close(got.float(), general.float(), rtol=ulp, atol=6e-5)


@pytest.mark.parametrize("d", [64, 96])
def test_planned_layers_match_per_call_lists(device, d):
    q, k, v, cache, md = build_case(device, torch.bfloat16, LENGTHS, QLENS, 8, 2, d, 16, seed=d)
    expected = operator()(q, k, v, cache, md)
    plan = AttentionPlan(md, 8, cache)
    for _ in range(2):
        assert torch.equal(hip_attention_over_cache(q, cache, md, plan=plan), expected)


def test_workspace_too_small_takes_the_any_shape_kernel(device):
    """The any-shape kernel needs no workspace; a caller that passes none at
    head_dim 64 is still answered."""

    import math

    from micro_vllm_amd import _native
    from micro_vllm_amd.attention.operators.mi355x_paged import batch_descriptor

    q, k, v, cache, md = build_case(device, torch.bfloat16, LENGTHS, QLENS, 8, 2, 64, 16, seed=1)
    expected = operator()(q, k, v, cache, md)
    out = torch.empty_like(q)
    batch, keep = batch_descriptor(md, device)
    _native.check(
        _native.load().mvllm_paged_attention(
            _native.tensor3(q), _native.kv_cache(cache), batch, _native.tensor3(out), 1.0 / math.sqrt(64), None, 0,
            _native.stream_handle(device),
        ),
        "mvllm_paged_attention",
    )
    del keep
    torch.testing.assert_close(out.float(), expected.float(), rtol=2.0**-7, atol=6e-5)
