"""The BF16 block's LayerNorm and bias heads, two rows per wave pass: odd and
even row counts of a tile, rows of very different means in one pass, and an
affine LayerNorm, against the FP32 oracle on the same bf16-rounded inputs
within 2e-2 of its largest value (BF16 storage rounds each stage to 2^-9).  The
workspace holds NaN: key tiles past the last key are not projected (N = 97 of
128, 130 of 256), and nothing may read them.
"""
from __future__ import annotations

import pytest
import torch

from fireprot_amd import block as hip_block
from fireprot_amd import workloads
from oracle import triangle_attention as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 31, 33, 63, 97, 130])
@pytest.mark.parametrize("ending", [False, True])
def test_rows_of_one_pass_do_not_mix(n, ending):
    print(f"case n={n} ending={ending}", flush=True)
    z = workloads.make_pair(n)
    # neighbouring rows (along either axis) with means 0 and 16, scales 1 and 1/8
    parity = ((torch.arange(n)[:, None] + torch.arange(n)[None, :]) % 2).float()[..., None]
    z = (z * (1.0 - 0.875 * parity) + 16.0 * parity).bfloat16()
    w = workloads.make_weights(bias_scale=4.0)
    w["ln_w"] = 1.0 + 0.25 * torch.sin(torch.arange(128.0))
    w["ln_b"] = 0.1 * torch.cos(torch.arange(128.0))
    w = {k: v.bfloat16() if isinstance(v, torch.Tensor) else v for k, v in w.items()}
    w32 = {k: v.float() if isinstance(v, torch.Tensor) else v for k, v in w.items()}
    expected = oracle.block(z.float(), None, oracle.BlockParams(**w32), ending=ending)
    ws = torch.full((hip_block.workspace_bytes(n, torch.bfloat16) // 4,), float("nan"),
                    device="cuda").view(torch.uint8)
    with torch.inference_mode():
        actual = hip_block.triangle_attention_block(
            z.cuda(), None, hip_block.BlockWeights.from_tensors(**w, dtype=torch.bfloat16).to("cuda"),
            ending=ending, workspace=ws).float().cpu()
    if ending:
        actual, expected = actual.transpose(0, 1), expected.transpose(0, 1)
    assert (actual - expected).abs().max() <= 2e-2 * expected.abs().max()
