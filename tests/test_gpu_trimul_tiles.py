"""The triangle multiplication at the sizes where its projection's work split
changes, and where the contraction's keys end inside a 128-key panel.

On 256 CUs the projection deals whole rows (N = 33, 96, 160, 256, 353, 362, 363),
or tiles of all rows with atomic row maxima (N = 97, 128, 129, 257, 300, 352, the
largest); N = 33, 97, 129, 257 and 353 end a key run of 32 after one key.  Sampled rows are held to
float64: the largest error within twice that of the same oracle in FP32 (or
2e-6 of the largest value).  The workspace holds NaN, so a maximum or a tile
left unwritten shows.
"""
from __future__ import annotations

import pytest
import torch

from fireprot_amd import triangle_multiplication as htm
from fireprot_amd import workloads
from oracle import triangle_multiplication as tm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [33, 96, 97, 128, 129, 160, 256, 257, 300, 352, 353, 362, 363])
@pytest.mark.parametrize("outgoing", [True, False])
def test_work_split_edges(n, outgoing):
    print(f"case n={n} outgoing={outgoing}", flush=True)
    z = workloads.make_pair(n)
    mask = workloads.make_mask(n, n - n // 7)
    w = workloads.make_trimul_weights(affine=True, biases=True)
    p = tm.TriMulParams(**w)
    p64 = tm.TriMulParams(**{k: None if v is None else v.double() for k, v in w.items()})
    rows = torch.tensor(sorted({0, 1, n // 2, n - n // 7 - 1, n - 1}))
    ref32 = tm.update(z, mask, p, outgoing=outgoing, rows=rows).double()
    ref64 = tm.update(z.double(), mask.double(), p64, outgoing=outgoing, rows=rows)
    ws = torch.full((htm.workspace_bytes(n) // 4,), float("nan"), device="cuda").view(torch.uint8)
    wt = htm.TriMulWeights.from_tensors(**w).to("cuda")
    with torch.inference_mode():
        out = htm.triangle_multiplication(z.cuda(), mask.cuda(), wt, outgoing=outgoing,
                                          workspace=ws)
        again = htm.triangle_multiplication(z.cuda(), mask.cuda(), wt, outgoing=outgoing,
                                            workspace=ws)
    assert torch.equal(out, again)
    err = (out[rows.cuda()].cpu().double() - ref64).abs().max().item()
    bar = max(2e-6 * ref64.abs().max().item(), 2.0 * (ref32 - ref64).abs().max().item())
    assert err <= bar, (err, bar)
