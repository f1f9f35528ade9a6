"""A plan made over one cache and a layer whose cache differs: the layer is
answered through lists of its own, and the plan stays good for its own layers.

The decode splits, the counters of finished splits and the query blocks all
follow from the KV heads, head_dim and element type, so lists made for other
ones would leave requests unfinished.
"""

from __future__ import annotations

import pytest
import torch

from micro_vllm_amd.attention.operators.mi355x_paged import AttentionPlan, hip_attention_over_cache, plan_geometry


def cache(blocks=4, block=16, heads=8, dim=128, dtype=torch.bfloat16):
    return torch.zeros((2, blocks, block, heads, dim), dtype=dtype)


def test_geometry_ignores_what_the_lists_do_not_depend_on():
    c = cache()
    assert plan_geometry(c) == plan_geometry(torch.ones_like(c)) == plan_geometry(cache(blocks=9))


@pytest.mark.parametrize(
    "other",
    [
        cache(heads=1),
        cache(heads=16),
        cache(dim=64),
        cache(block=32),
        cache(dtype=torch.float16),
        cache(dtype=torch.float32),
        torch.zeros((2, 4, 16, 8, 256), dtype=torch.bfloat16)[..., :128],
        torch.zeros(cache().numel() + 1, dtype=torch.bfloat16)[1:].view(cache().shape),
        torch.zeros(2 * 9 * 16 * 8 * 128, dtype=torch.bfloat16).as_strided((2, 4, 16, 8, 128), (65537, 16384, 1024, 128, 1)),
    ],
    ids=["1-head", "16-heads", "dim-64", "block-32", "fp16", "fp32", "strided", "misaligned", "odd-plane"],
)
def test_geometry_tells_caches_apart(other):
    assert plan_geometry(cache()) != plan_geometry(other)


@pytest.mark.gpu
@pytest.mark.parametrize("planned", [(128, 1), (128, 8), (128, 2), (64, 2), "fp32"], ids=str)
@pytest.mark.parametrize("qlens", [[1, 1, 1, 1, 1], [1, 40, 1, 17, 1]], ids=["decode", "mixed"])
def test_a_layer_of_another_geometry_is_answered(device, planned, qlens):
    from test_gpu_attention import build_case, operator

    lengths = [3000, 700, 5, 1200, 64]
    q, k, v, layer_cache, md = build_case(device, torch.bfloat16, lengths, qlens, 16, 4, 128, 16, seed=4)
    expected = operator()(q, k, v, layer_cache, md)
    dim, heads, dtype = (128, 4, torch.float32) if planned == "fp32" else (*planned, torch.bfloat16)
    other = torch.randn((*layer_cache.shape[:3], heads, dim), device=device).to(dtype)
    plan = AttentionPlan(md, 16, other)
    q_other = torch.ones((q.shape[0], 16, dim), dtype=dtype, device=device)
    own = hip_attention_over_cache(q_other, other, md)
    for _ in range(2):
        assert torch.equal(hip_attention_over_cache(q, layer_cache, md, plan=plan), expected)
        assert torch.equal(hip_attention_over_cache(q_other, other, md, plan=plan), own)
