"""SwiGLU on 16-byte rows: bit for bit against the element-wise form.

A 4-byte aligned input (and a row of fewer than 512 elements) takes the kernel that evaluates the library's
exponential and the IEEE division; 16-byte aligned rows take the vector
kernel. The two agree to an fp32 ulp or so before the rounding to 16 bits, so
at most a handful of the 65,536 gate values land on the other side of a
rounding boundary (one unit in the last place); zeros keep their sign.
"""

from __future__ import annotations

import pytest
import torch

from micro_vllm_amd import layers

pytestmark = pytest.mark.gpu


def element_wise(gate_up):
    shifted = torch.empty(gate_up.numel() + 2, dtype=gate_up.dtype, device=gate_up.device)[2:].view(gate_up.shape)
    shifted.copy_(gate_up)
    assert shifted.data_ptr() % 16 != 0
    return layers.silu_mul(shifted)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("factor", [1.0, -0.7])
def test_every_gate_value(device, dtype, factor):
    gate = torch.arange(65536, device=device, dtype=torch.int32).to(torch.int16).view(dtype).view(1, -1)
    gate_up = torch.cat([gate, torch.full_like(gate, factor)], 1).contiguous()
    got, expected = layers.silu_mul(gate_up), element_wise(gate_up)
    nan = torch.isnan(expected)
    assert torch.equal(torch.isnan(got), nan)
    step = (got.view(torch.int16).int() - expected.view(torch.int16).int()).abs()[~nan]
    assert int(step.max()) <= 1 and int((step != 0).sum()) <= 4


@pytest.mark.parametrize(("rows", "inter"), [(1, 8), (3, 504), (3, 512), (3, 1024), (5, 1032), (257, 3072), (1171, 14336)])
def test_row_and_column_remainders(device, rows, inter):
    """Odd row counts, row widths that end inside a workgroup, and a padded row
    stride."""

    wide = torch.randn((rows, 2 * inter + 16), device=device).to(torch.bfloat16)
    gate_up = wide[:, : 2 * inter]
    gate, up = gate_up.float().chunk(2, dim=-1)
    expected = (gate / (1 + torch.exp(-gate))).to(torch.bfloat16).float() * up
    # Half a unit in the last place of the product's rounding (2^-9 relative) and of the gate's (a full one where
    # the two exponentials straddle a rounding boundary: 2^-8).
    torch.testing.assert_close(layers.silu_mul(gate_up).float(), expected, rtol=2.0**-8 + 2.0**-9, atol=1e-30)
