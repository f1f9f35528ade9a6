"""Decode splits chosen on the device, and the merge inside the split kernel.

Batches at the ends of the rule that picks the split length (every request at
the table's full reach, so the work list is as full as it gets; one long
context beside many short ones; more requests than the list builder's
threads; contexts around the shortest split), and at every size of merge
round (up to 2, 4, 8, 16, 24, 32 and more splits: the two "merge-rounds" batches
give 1-2, 4, 8, 12, 16 and 32 and 5, 11, 21, 23 and 30 on 256 CUs, "one-long" 40),
against the oracle.
"""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest
import torch

from micro_vllm_amd.attention import SlidingWindowSpec
from micro_vllm_amd.attention.operators.mi355x_paged import AttentionPlan, hip_attention_over_cache
from test_gpu_attention import build_case, operator, run_and_check

pytestmark = pytest.mark.gpu

BATCHES = {
    "full-reach": [2048] * 64,
    "full-reach-short": [193] * 300,
    "one-long": [20_000] + [3, 50] * 40,
    "many-requests": [1 + (37 * i) % 400 for i in range(1100)],
    "around-the-shortest-split": [191, 192, 193, 207, 208, 209, 383, 384, 385],
    "merge-rounds": [300, 700, 1500, 3000, 4500, 6100, 12_000],
    "merge-rounds-short": [300, 700, 1300, 1450, 1900],
    "single": [6145],
    "whole-even": [1000 + r % 20 for r in range(110)],
    "whole-short": [1 + (r * 7) % 320 for r in range(200)],
}


@pytest.mark.parametrize("name", sorted(BATCHES))
@pytest.mark.parametrize(("hq", "hkv"), [(4, 2), (5, 5)], ids=["gqa", "mha-5"])
@pytest.mark.parametrize("hint", [True, False], ids=["hint", "no-hint"])
def test_split_rule_ends(device, name, hq, hkv, hint):
    lengths = BATCHES[name]
    q, k, v, cache, md = build_case(device, torch.bfloat16, lengths, [1] * len(lengths), hq, hkv, 128, 16, seed=hq)
    if hint:
        md = dataclasses.replace(md, max_query_len=1)
    run_and_check(q, k, v, cache, md, torch.bfloat16)


@pytest.mark.parametrize("d", [64, 128])
def test_beside_prefill_work(device, d):
    lengths = [9000, 4000, 300, 256, 257, 700, 60] + [1024] * 20
    qlens = [1, 1, 1, 1, 1, 200, 60] + [1] * 20
    q, k, v, cache, md = build_case(device, torch.float16, lengths, qlens, 8, 2, d, 32, seed=d,
                                    spec=SlidingWindowSpec(3000))
    run_and_check(q, k, v, cache, md, torch.float16)


def test_merge_counters_return_to_zero_between_layers(device):
    """One plan, several layers and graph replays: every launch finds the
    counters of finished splits at zero, whichever workgroup came last."""

    lengths = [6100, 900, 192, 5, 3000]
    q, k, v, cache, md = build_case(device, torch.bfloat16, lengths, [1] * 5, 16, 8, 128, 16, seed=9)
    expected = operator()(q, k, v, cache, md)
    plan = AttentionPlan(md, 16, cache)
    for _ in range(4):
        assert torch.equal(hip_attention_over_cache(q, cache, md, plan=plan), expected)
    side = torch.cuda.Stream(device)
    side.wait_stream(torch.cuda.current_stream(device))
    with torch.cuda.stream(side):
        hip_attention_over_cache(q, cache, md, plan=plan)
    torch.cuda.current_stream(device).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        first = hip_attention_over_cache(q, cache, md, plan=plan)
        second = hip_attention_over_cache(q, cache, md, plan=plan)
    for _ in range(4):
        first.zero_()
        second.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(first, expected) and torch.equal(second, expected)
        assert torch.equal(hip_attention_over_cache(q, cache, md, plan=plan), expected)


def test_rows_that_no_split_writes(device):
    """A decode request with nothing visible is NaN, tokens after the last
    request are zero, and the requests around them are answered."""

    lengths = [500, 40, 300]
    q, k, v, cache, md = build_case(device, torch.bfloat16, lengths, [1, 1, 1], 16, 8, 128, 16, seed=2)
    expected = operator()(q, k, v, cache, md)
    pad = lambda t, n, value: torch.cat([t, torch.full((n, *t.shape[1:]), value, dtype=t.dtype, device=device)])  # noqa: E731
    starts = md.query_context_start_positions.clone()
    starts[1] = md.query_positions[1] + 1
    md = dataclasses.replace(
        md,
        query_positions=pad(md.query_positions, 20, 0),
        query_context_start_positions=pad(starts, 20, 0),
        slot_mapping=pad(md.slot_mapping, 20, -1),
        max_query_len=1,
    )
    out = operator()(pad(q, 20, 1.0), pad(k, 20, 1.0), pad(v, 20, 1.0), cache, md)
    assert torch.equal(out[[0, 2]], expected[[0, 2]])
    assert torch.isnan(out[1]).all() and (out[3:] == 0).all()
