"""The pair transition at the row counts where its tiling changes.

With C compute units a call takes small tiles (32 rows a work-group, then 64)
up to 64 C rows, half tiles (128 rows) up to 128 C, full tiles (256 rows)
above, and whole rounds of full tiles followed by one of these for the rows
left over.  Every row is held to float64: the largest error stays within twice
that of the same expression in FP32 torch (or 2e-6 of the largest value).
"""
from __future__ import annotations

import pytest
import torch

from fireprot_amd import transition as htr
from fireprot_amd import workloads

pytestmark = pytest.mark.gpu


def _reference(z, w, dtype):
    w = {k: v.to("cuda", dtype) for k, v in w.items() if v is not None}
    out = torch.empty_like(z)
    for at in range(0, len(z), 1 << 15):
        x = torch.nn.functional.layer_norm(z[at:at + (1 << 15)].to(dtype), (128,), w["ln_w"],
                                           w["ln_b"], 1e-5)
        h = torch.nn.functional.silu(x @ w["w_a"].t()) * (x @ w["w_b"].t())
        out[at:at + (1 << 15)] = (h @ w["w_o"].t()).to(out.dtype)
    return out


@pytest.mark.parametrize("per_cu,extra", [(0, 1), (0, 33), (32, 0), (32, 1), (64, 0), (64, 1),
                                          (128, -1), (128, 1), (256, 0), (256, 1), (288, 1),
                                          (320, 1), (384, 1)])
def test_rows_at_the_edges_of_the_tile_modes(per_cu, extra):
    rows = per_cu * torch.cuda.get_device_properties(0).multi_processor_count + extra
    print(f"case rows={rows}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows)
    z = torch.randn(rows, 128, generator=g, device="cuda") * 2.0 + 0.5
    w = workloads.make_transition_weights(affine=True)
    wt = htr.TransitionWeights.from_tensors(**w).to("cuda")
    with torch.inference_mode():
        out = htr.transition(z, wt)
        again = htr.transition(z, wt)
        target = z.clone().view(1, rows, 128)
        htr.pair_transition_residual(target, wt)
        ref64 = _reference(z.double(), w, torch.float64)
        err32 = (_reference(z, w, torch.float32).double() - ref64).abs().max().item()
        err = (out.double() - ref64).abs().max().item()
        bar = max(2e-6 * ref64.abs().max().item(), 2.0 * err32)
    assert err <= bar, (err, err32)
    assert torch.equal(out, again)
    assert torch.equal(target.view(rows, 128), z + out)  # the residual adds the rounded update
