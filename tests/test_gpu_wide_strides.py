"""A cache whose tokens lie 256 MiB apart: decodes at head_dim 128 take the
general split kernel, which addresses rows in 64 bits, bit for bit; chunks, which
no matrix-core kernel takes there, agree with the oracle."""

from __future__ import annotations

import pytest
import torch

from test_gpu_attention import build_case, operator, run_and_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qlens", [[1, 1, 1, 1], [1, 3, 1, 1]], ids=["decodes", "mixed"])
def test_tokens_far_apart(device, monkeypatch, qlens):
    q, k, v, cache, md = build_case(device, torch.bfloat16, [40, 33, 17, 90], qlens, 8, 2, 128, 16, seed=4)
    planes, blocks, block, heads, dim = cache.shape
    token, plane, page = 2**27, heads * dim, 2 * heads * dim
    memory = torch.empty((block - 1) * token + blocks * page, dtype=cache.dtype, device=device)
    wide = memory.as_strided(cache.shape, (plane, page, token, dim, 1))
    wide.copy_(cache)
    got = run_and_check(q, k, v, wide, md, torch.bfloat16)
    monkeypatch.setenv("MVLLM_DECODE_KERNEL", "general")
    expected = operator()(q, k, v, cache, md)
    decodes = [t for t, n in enumerate(n for n in qlens for _ in range(n)) if n == 1]
    assert torch.equal(got[decodes], expected[decodes])
