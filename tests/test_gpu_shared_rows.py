"""Padding rows whose attention weights are formed once for the whole call.

A row whose every key carries the mask bias m = -1e9 has the logits
fl(fl(s + m) + bias) = fl(m + bias) whatever its products s, while |s| stays
below half the float32 spacing of m (32).  The prepare stage bounds |s| by the
row's own 2-norms (words 2 and 3 of part 3 of its tile flags: max |q|^2 and
max |k|^2), which holds on rows for which 32 max|q| max|k| over the whole pair
does not; such rows run in the fast launch on the shared weights.
"""
from __future__ import annotations

import pytest
import torch

from fireprot_amd import block as hip_block
from fireprot_amd import workloads
from oracle import triangle_attention as oracle
from tests.helpers import hip_weights
from tests.test_gpu_fp32_accuracy import _check_regions
from tests.test_gpu_planes import _offsets

pytestmark = pytest.mark.gpu


# one key tile, a second, an odd and an even number of tiles, query rows past n
@pytest.mark.parametrize("n,valid", [(1, 0), (20, 17), (33, 30), (96, 64), (128, 127), (160, 130)])
@pytest.mark.parametrize("ending", [False, True])
def test_rows_inside_the_norm_bound_only(n, valid, ending):
    z = workloads.make_pair(n)
    mask = workloads.make_mask(n, valid)
    w = workloads.make_weights(bias_scale=4.0)
    w["w_q"], w["w_k"] = w["w_q"] * 3.0, w["w_k"] * 3.0
    print(f"case n={n} valid={valid} ending={ending}", flush=True)
    ws = torch.empty(hip_block.workspace_bytes(n), dtype=torch.uint8, device="cuda")
    with torch.inference_mode():
        out = hip_block.triangle_attention_block(z.cuda(), mask.cuda(), hip_weights(w),
                                                 ending=ending, workspace=ws)
        actual = (out.transpose(0, 1) if ending else out).cpu()
    at = _offsets(n)["flags"]
    words = ws[at:at + (16 * n + 6) * 4].cpu().view(torch.float32)
    flags, record = words[:16 * n].view(n, 4, 4), words[16 * n:]

    # the norms: at least the float64 ones, and within 2^-8 of them
    x = z.double().transpose(0, 1) if ending else z.double()
    y = oracle.layer_norm(x, w["ln_w"].double(), w["ln_b"].double())
    for word, name, scale in ((2, "w_q", 32 ** -0.5), (3, "w_k", 1.0)):
        v = (y @ w[name].double().t() * scale).view(n, n, 4, 32)
        norm2 = (v * v).sum(-1).amax((1, 2))
        ratio = flags[valid:, 3, word].double() / norm2[valid:]
        assert ratio.min() >= 1.0 and ratio.max() <= 1.0 + 2.0 ** -8, (name, ratio)
        assert (flags[:valid, 3, word] == 0).all()  # not formed on other rows
    bound = (flags[valid:, 3, 2] * flags[valid:, 3, 3]).sqrt().max().item()
    assert bound < 31.0, bound
    if n >= 20:  # the element bound alone would send these rows to the exact softmax
        assert 32.0 * record[0].item() * record[1].item() > 33.0
    _check_regions(f"n={n} ending={ending}", actual, z, mask, w, ending, torch.arange(n), valid)
