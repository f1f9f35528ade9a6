"""head_dim 64 and 96 (bf16 / fp16): values of V that are not finite, against the
any-shape kernel, which a query view that is not 16-byte aligned still takes."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from micro_vllm_amd.attention import ChunkedLocalSpec, SlidingWindowSpec
from test_gpu_attention import build_case, operator

pytestmark = pytest.mark.gpu

LENGTHS = [1, 17, 65, 700, 129, 600, 90, 1100]
QLENS = [1, 1, 1, 1, 100, 600, 3, 33]


def shifted(q):
    out = torch.empty(q.numel() + 1, dtype=q.dtype, device=q.device)[1:].view(q.shape)
    out.copy_(q)
    assert out.data_ptr() % 16 != 0
    return out


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 96])
@pytest.mark.parametrize("spec", [None, SlidingWindowSpec(100), ChunkedLocalSpec(48)], ids=repr)
def test_values_that_are_not_finite_reach_only_rows_that_see_them(device, bad, dtype, d, spec):
    """Rows of a workgroup share V tiles. A non-finite value of a chunk's own
    token stays out of the earlier tokens, and one in a decode's or chunk's
    history out of rows whose window has passed it; an infinity stays one. The
    bound is that of finite values: one unit in the last place and 2^-17 of the
    largest |v|."""

    q, k, v, cache, md = build_case(device, dtype, LENGTHS, QLENS, 8, 2, d, 16, spec=spec, seed=d)
    first = np.concatenate([[0], np.cumsum(QLENS)])
    v[first[4] + 40, 0, 5] = bad
    v[first[5] + 300, 1, d - 1] = bad
    v[first[5] + 599, 0, 0] = bad
    for r, position in ((3, 690), (7, 1062)):  # in the history of a decode and of a chunk
        block = int(md.block_table[r, position // 16])
        cache[1, block, position % 16, 0, 17] = bad
    expected = operator()(shifted(q), k, v, cache.clone(), md)
    got = operator()(q, k, v, cache, md)
    assert not torch.isfinite(expected).all()
    assert torch.isfinite(expected[first[4] : first[4] + 40]).all()
    assert torch.isfinite(expected[first[5] : first[5] + 300]).all()
    ulp = 2.0**-7 if dtype == torch.bfloat16 else 2.0**-10
    torch.testing.assert_close(got.float(), expected.float(), rtol=ulp, atol=6e-5, equal_nan=True)
