"""``fpx_attn_core_masked`` on finite operands of wide range, against plain torch
in float64: what an fp16 plane pair cannot hold beside a much larger value of
the same wave, tile or row must not be lost.

Bar, per output row (a query's 32 channels of a head) and per output channel
(all queries of a head): the largest error within max(2e-6 of the largest
sum_k w_k |v_k|, the scale at which FP32 rounds the sum; twice the largest error
of the same expression in FP32 torch).  2e-6 is the bar of the unit-scale cases
(16 ulp).  Where a key outside a row's softmax holds the large value, FP32
arithmetic multiplies it by exactly 0, so it does not count in that scale.
"""
from __future__ import annotations

import pytest
import torch

from tests.test_gpu_core_split import _inputs, _run, _torch

pytestmark = pytest.mark.gpu


def _check(q, k, v, bias, mask=None):
    out = _run(q, k, v, bias, mask).double()
    ref = _torch(q, k, v, bias, mask, torch.float64)
    low = _torch(q, k, v, bias, mask, torch.float32).double()
    size = _torch(q, k, v.abs(), bias, mask, torch.float64)
    assert torch.isfinite(ref).all()
    for dim in (3, 1):  # over a row's channels; over a channel's queries
        err, base = (out - ref).abs().amax(dim), (low - ref).abs().amax(dim)
        bar = torch.maximum(2e-6 * size.amax(dim), 2.0 * base)
        worst = (err / bar.clamp_min(1e-300)).max().item()
        assert worst <= 1.0, (dim, worst, err.max().item())


def _mask(batch, n, *keys):
    mask = torch.zeros(batch, n, device="cuda")
    mask[:, list(keys)] = -1e9
    return mask


@pytest.mark.parametrize("value", [1e4, 1e6, 1e9, 1e12, 1e30])
@pytest.mark.parametrize("key", [0, 70, 155])
def test_value_of_a_masked_key(key, value):
    n = 156
    q, k, v, bias = _inputs(2, n, 21)
    v[:, key] = value
    _check(q, k, v, bias, _mask(2, n, key))


@pytest.mark.parametrize("value", [1e6, 1e10, 1e14])
def test_value_of_a_key_of_small_weight(value):
    n = 100
    q, k, v, bias = _inputs(2, n, 22)
    v[:, 40] *= value
    bias[:, :, 40] = -60.0
    _check(q, k, v, bias)


@pytest.mark.parametrize("gain", [1e4, 1e8, 1e10])
@pytest.mark.parametrize("which", ["q", "k"])
def test_one_row_far_above_the_others_of_its_tile(which, gain):
    """A query's logits grow alone; a key's are cut off by its bias."""
    n = 132
    q, k, v, bias = _inputs(2, n, 23)
    {"q": q, "k": k}[which][:, 37] *= gain
    if which == "k":
        bias[:, :, 37] = -100.0 * gain
    _check(q, k, v, bias)


@pytest.mark.parametrize("gain", [1e4, 1e8])
@pytest.mark.parametrize("which", ["q", "k"])
def test_one_channel_far_above_the_others(which, gain):
    """The channel's partner is 0, so the other channels make the logits."""
    n = 64
    q, k, v, bias = _inputs(2, n, 24)
    big, zero = (q, k) if which == "q" else (k, q)
    big[..., 5] *= gain
    zero[..., 5] = 0.0
    _check(q, k, v, bias)


@pytest.mark.parametrize("gain", [1e-12, 1e-8, 1e-4, 1e4, 1e8])
def test_one_value_channel_at_another_scale(gain):
    n = 132
    q, k, v, bias = _inputs(2, n, 25)
    v[:, :, 2, 9] *= gain
    _check(q, k, v, bias)


@pytest.mark.parametrize("gain", [1e6, 1e9])
def test_query_that_attends_only_small_values(gain):
    """Half of the keys hold values `gain` times the others'; some queries
    see only the others."""
    n = 160
    q, k, v, bias = _inputs(2, n, 26)
    v[:, 80:] *= gain
    bias[:, ::7, 80:] = -200.0
    _check(q, k, v, bias)


@pytest.mark.parametrize("value", [1e6, 1e10])
def test_fully_masked_row_with_a_wide_value_range(value):
    """All keys masked alike: every weight counts, one key is cut off by its bias."""
    n = 100
    q, k, v, bias = _inputs(2, n, 27)
    mask = torch.zeros(2, n, device="cuda")
    mask[1] = -1e9
    v[:, 33] *= value
    bias[:, :, 33] = -1e6
    q[1] = 0.0  # logits tie on the grid of 64 that the mask sets, in float64 too
    bias[..., torch.arange(n, device="cuda") != 33] = 0.0
    _check(q, k, v, bias, mask)


@pytest.mark.parametrize("gain", [1.0, 4.0, 16.0, 64.0])
def test_logit_scales(gain):
    """Logits of up to 64 standard deviations of q k: within twice the largest
    error of FP32 torch, or 2e-6 of the largest value."""
    n = 260
    q, k, v, bias = _inputs(2, n, 28)
    q, bias = q * gain, bias * gain
    out = _run(q, k, v, bias).double()
    ref = _torch(q, k, v, bias, None, torch.float64)
    low = _torch(q, k, v, bias, None, torch.float32).double()
    err, base = (out - ref).abs().max().item(), (low - ref).abs().max().item()
    print(f"gain {gain}: err {err:.3e}, FP32 torch {base:.3e}", flush=True)
    assert err <= max(2e-6 * ref.abs().max().item(), 2.0 * base), (err, base)


@pytest.mark.parametrize("ratio", [16.0, 60.0, 250.0, 4000.0])
@pytest.mark.parametrize("n", [260, 1536])
def test_many_equal_small_weights_on_large_values(n, ratio):
    """One key takes nearly all weight, the others share one tiny weight on
    values `ratio` times its own: equal terms round alike, so errors add up
    instead of averaging out, n times half an ulp in an FP32 sum of n terms
    (the bar's 2^-24: a sum between the powers of two)."""
    q, k, v, bias = _inputs(1, n, 29)
    q.zero_()
    v.fill_(ratio)
    v[:, 7] = 1.0
    bias.zero_()
    for i, drop in enumerate((14.0, 16.5, 18.3, 19.7)):  # weights of 2^-20 to 2^-28
        bias[i] = -drop
    bias[:, :, 7] = 0.0
    out = _run(q, k, v, bias).double()
    ref = _torch(q, k, v, bias, None, torch.float64)
    worst = ((out - ref).abs() / ref.abs()).max().item()
    print(f"n {n} ratio {ratio}: {worst:.2e}", flush=True)
    assert worst <= n * 2.0 ** -24, worst
