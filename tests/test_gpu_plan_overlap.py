"""Planned calls of one plan that overlapped spoil themselves at most: the
counters of finished splits come back to zero whatever the interleaving, so that
later calls on the plan are answered."""

from __future__ import annotations

import pytest
import torch

from micro_vllm_amd.attention.operators.mi355x_paged import AttentionPlan, hip_attention_over_cache
from test_gpu_attention import build_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [16, 24], ids=["pipelined", "general"])
def test_calls_after_an_overlap_are_answered(device, block):
    """The overlapping calls are alike, so they write the same partials; only the
    order in which the workgroups of both count is open."""

    lengths = [500 + 7 * r for r in range(60)]
    q, k, v, cache, md = build_case(device, torch.bfloat16, lengths, [1] * 60, 16, 8, 128, block, seed=3, nan_cache=False)
    plan = AttentionPlan(md, 16, cache)
    streams = [torch.cuda.Stream(device) for _ in range(2)]
    gen = torch.Generator(device=device).manual_seed(1)
    for _ in range(10):
        torch.cuda.synchronize()
        for _ in range(10):
            for stream in streams:
                with torch.cuda.stream(stream):
                    hip_attention_over_cache(q, cache, md, plan=plan)
        torch.cuda.synchronize()
        other = torch.randn(q.shape, generator=gen, device=device).to(q.dtype)
        assert torch.equal(hip_attention_over_cache(other, cache, md, plan=plan), hip_attention_over_cache(other, cache, md))
