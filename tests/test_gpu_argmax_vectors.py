"""Greedy sampling on 16-byte rows: the two-level search against torch.argmax.

Widths around the workgroup's rounds (1,024 lanes, four vectors of 16 bytes
each), fewer vectors than lanes, tails past the last whole vector; ties
within a vector, between vectors of a lane and between lanes; a NaN in the
tail only, and in a vector that also holds the row's largest number.
"""

from __future__ import annotations

import pytest
import torch

from micro_vllm_amd import layers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("vectors", [1, 2, 1023, 1025, 3999, 4000, 4097, 8192, 16_001])
@pytest.mark.parametrize("tail", [0, 3])
@pytest.mark.parametrize("rows", [12, 401], ids=["few", "many"])
def test_widths_ties_and_nan(device, dtype, vectors, tail, rows):
    """12 rows of 4,000 vectors or more (fp32: 16,000) take the two-level search,
    401 rows and narrower ones the element-wise one."""
    per = 4 if dtype == torch.float32 else 8
    cols = vectors * per + tail
    gen = torch.Generator(device=device).manual_seed(cols)
    stride = (vectors + 1) * per  # rows stay 16-byte aligned
    logits = torch.empty((rows, stride), dtype=dtype, device=device)[:, :cols]
    logits.copy_(torch.randint(-300, 300, (rows, cols), generator=gen, device=device).to(dtype) / 64)
    assert logits.data_ptr() % 16 == 0 and logits.stride(0) * logits.element_size() % 16 == 0
    logits[1] = 2.0  # every entry ties
    logits[2, [cols - 1, cols // 2, cols // 3]] = 9.0
    logits[3] = float("-inf")
    logits[4] = float("-inf")
    logits[4, cols - 1] = -30_000.0
    logits[5, cols - 1] = float("nan")
    logits[6, cols // 2] = float("nan")
    logits[6, max(0, cols // 2 - 1)] = float("inf")
    logits[7] = float("nan")
    logits[8] = -0.0
    logits[8, cols // 2] = 0.0
    logits[9] = -(logits[9].abs() + 1)
    logits[10, cols // 2] = -float("nan")
    assert torch.equal(layers.argmax_rows(logits), torch.argmax(logits, dim=-1))
