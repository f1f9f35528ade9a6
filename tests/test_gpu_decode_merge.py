"""Decode batches by head layout: the partials merged by the workgroup that
finishes a request, or by a launch of its own (more than two query heads per KV
head, one KV head), and the split lengths that follow from the KV heads, against
the oracle."""

from __future__ import annotations

import dataclasses

import pytest
import torch

from micro_vllm_amd.attention import SlidingWindowSpec
from micro_vllm_amd.attention.operators.mi355x_paged import AttentionPlan, hip_attention_over_cache
from test_gpu_attention import build_case, operator, run_and_check

pytestmark = pytest.mark.gpu

# One to two splits, every size of merge round and two rounds (17,000 tokens in
# splits of about 272), and requests that are not split.
LENGTHS = [1, 64, 65, 130, 260, 700, 1300, 1700, 3000, 17_000]


@pytest.mark.parametrize(("hq", "hkv"), [(1, 1), (2, 1), (3, 1), (9, 1), (16, 1), (6, 2), (14, 2), (9, 3), (20, 4), (15, 5), (32, 8)], ids=str)
@pytest.mark.parametrize("hint", [1, None, 2], ids=["decodes", "no-hint", "maybe-chunks"])
def test_head_layouts(device, hq, hkv, hint):
    """Odd head counts leave a wave of the merge one head or none; with the hint
    that chunks may come, groups of up to eight are merged in the split kernel."""

    q, k, v, cache, md = build_case(device, torch.bfloat16, LENGTHS, [1] * len(LENGTHS), hq, hkv, 128, 16, seed=hq)
    run_and_check(q, k, v, cache, dataclasses.replace(md, max_query_len=hint), torch.bfloat16)


@pytest.mark.parametrize("d", [64, 96, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("hq", "hkv", "bs"), [(12, 2, 16), (16, 1, 48), (40, 4, 24)], ids=str)
def test_dims_and_the_general_kernel(device, d, dtype, hq, hkv, bs):
    """Block sizes that are not multiples of 16 take the general split kernel at
    head_dim 128 (and no splits at all below)."""

    q, k, v, cache, md = build_case(device, dtype, LENGTHS, [1] * len(LENGTHS), hq, hkv, d, bs, seed=d, spec=SlidingWindowSpec(9000))
    run_and_check(q, k, v, cache, md, dtype)


@pytest.mark.parametrize("longest", [20, 64, 65, 120, 128, 136])
@pytest.mark.parametrize("chunk", [0, 3])
@pytest.mark.parametrize(("hq", "hkv", "bs"), [(16, 8, 8), (14, 2, 24), (32, 32, 8)], ids=str)
def test_the_general_kernel_without_splits(device, longest, chunk, hq, hkv, bs):
    """Tables that reach at most 128 tokens: no request is split and no merge launched."""

    lengths = [longest, 1, max(1, longest - 9)] * 20 + [longest] * (chunk > 0)
    qlens = [1] * 60 + [chunk] * (chunk > 0)
    q, k, v, cache, md = build_case(device, torch.bfloat16, lengths, qlens, hq, hkv, 128, bs, seed=longest)
    run_and_check(q, k, v, cache, dataclasses.replace(md, max_query_len=max(1, chunk)), torch.bfloat16)
    plan = AttentionPlan(md, hq, cache)
    assert torch.equal(hip_attention_over_cache(q, cache, md, plan=plan), hip_attention_over_cache(q, cache, md))


@pytest.mark.parametrize(("requests", "n"), [(40, 600), (190, 300), (200, 300), (33, 1500)])
@pytest.mark.parametrize(("hq", "hkv"), [(4, 1), (16, 4), (16, 16)], ids=str)
def test_batches_around_the_rules_ends(device, requests, n, hq, hkv):
    lengths = [n - (r * n) // (2 * requests) for r in range(requests)]
    q, k, v, cache, md = build_case(device, torch.float16, lengths, [1] * requests, hq, hkv, 128, 16, seed=n)
    run_and_check(q, k, v, cache, dataclasses.replace(md, max_query_len=1), torch.float16)


@pytest.mark.parametrize(("hq", "hkv"), [(16, 1), (14, 2), (28, 4)], ids=str)
def test_beside_chunks(device, hq, hkv):
    lengths = [17_000, 2000, 900, 64, 5] + [1024] * 30 + [300, 70]
    qlens = [1] * 35 + [200, 20]
    q, k, v, cache, md = build_case(device, torch.bfloat16, lengths, qlens, hq, hkv, 128, 16, seed=hq)
    run_and_check(q, k, v, cache, dataclasses.replace(md, max_query_len=200), torch.bfloat16)


def test_planned_layers_and_replays(device):
    """The plan holds the first partial row of each request; every planned call
    and replay merges by it."""

    q, k, v, cache, md = build_case(device, torch.bfloat16, LENGTHS, [1] * len(LENGTHS), 28, 4, 128, 16, seed=9)
    md = dataclasses.replace(md, max_query_len=1)
    expected = operator()(q, k, v, cache, md)
    plan = AttentionPlan(md, 28, cache)
    side = torch.cuda.Stream(device)
    side.wait_stream(torch.cuda.current_stream(device))
    with torch.cuda.stream(side):
        hip_attention_over_cache(q, cache, md, plan=plan)
    torch.cuda.current_stream(device).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        first = hip_attention_over_cache(q, cache, md, plan=plan)
        second = operator()(q, k, v, cache, md)
    for _ in range(4):
        first.zero_()
        second.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(first, expected) and torch.equal(second, expected)
        assert torch.equal(hip_attention_over_cache(q, cache, md, plan=plan), expected)


def test_rows_that_no_split_writes(device):
    q, k, v, cache, md = build_case(device, torch.bfloat16, [500, 400, 300], [1, 1, 1], 16, 1, 128, 16, seed=2)
    expected = operator()(q, k, v, cache, md)
    pad = lambda t, n, value: torch.cat([t, torch.full((n, *t.shape[1:]), value, dtype=t.dtype, device=device)])  # noqa: E731
    starts = md.query_context_start_positions.clone()
    starts[1] = md.query_positions[1] + 1  # the second request sees nothing
    md = dataclasses.replace(
        md, query_positions=pad(md.query_positions, 20, 0), query_context_start_positions=pad(starts, 20, 0),
        slot_mapping=pad(md.slot_mapping, 20, -1), max_query_len=1,
    )
    out = operator()(pad(q, 20, 1.0), pad(k, 20, 1.0), pad(v, 20, 1.0), cache, md)
    assert torch.equal(out[[0, 2]], expected[[0, 2]])
    assert torch.isnan(out[1]).all() and (out[3:] == 0).all()
