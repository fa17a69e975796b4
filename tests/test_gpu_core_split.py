"""``fpx_attn_core_masked`` splits its operands into fp16 planes tile by tile:
the cases where a plane exponent, a softmax reference or the plane form itself
has to give way, against plain torch in float64.

Bar: the largest error within max(2e-6 of the largest value, twice the error of
the same expression in FP32 torch); NaN and infinities where torch has them.
"""
from __future__ import annotations

import pytest
import torch

from fireprot_amd import _native

pytestmark = pytest.mark.gpu


def _inputs(batch, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn(batch, n, 4, 32, device="cuda", generator=g) for _ in range(3))
    return q / 32 ** 0.5, k, v, torch.randn(4, n, n, device="cuda", generator=g)


def _run(q, k, v, bias, mask=None, row=None):
    batch, n = q.shape[:2]
    out = torch.full_like(q, 7.0)
    _native.check(_native.library().fpx_attn_core_masked(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), None if mask is None else mask.data_ptr(),
        0 if mask is None else n, bias.data_ptr(), row or n, out.data_ptr(), batch, n,
        torch.cuda.current_stream().cuda_stream), "fpx_attn_core_masked")
    return out


def _torch(q, k, v, bias, mask, dtype):
    q, k, v = (t.to(dtype).permute(0, 2, 1, 3).contiguous() for t in (q, k, v))
    s = torch.matmul(q, k.transpose(2, 3).contiguous())
    if mask is not None:
        s = s + mask.to(dtype)[:, None, None, :]
    return torch.matmul(torch.softmax(s + bias.to(dtype), -1), v).permute(0, 2, 1, 3)


def _check(q, k, v, bias, mask=None):
    out = _run(q, k, v, bias, mask).double()
    ref = _torch(q, k, v, bias, mask, torch.float64)
    low = _torch(q, k, v, bias, mask, torch.float32).double()
    bar = max(2e-6 * ref.abs().max().item(), 2.0 * (low - ref).abs().max().item())
    err = (out - ref).abs().max().item()
    assert err <= bar, (err, bar)


@pytest.mark.parametrize("n", [4, 28, 32, 36, 64, 100, 128, 132, 260])
@pytest.mark.parametrize("masked", [False, True])
def test_tile_edges(n, masked):
    q, k, v, bias = _inputs(3, n, n)
    mask = None
    if masked:
        mask = 1e9 * ((torch.arange(n, device="cuda") % 3 != 1).float() - 1.0).repeat(3, 1)
    _check(q, k, v, bias, mask)


@pytest.mark.parametrize("which", ["q", "k", "v"])
@pytest.mark.parametrize("scales", [(1e-6, 1.0, 1e4), (1e4, 1.0, 1e-6), (0.0, 1.0, 0.0),
                                    (1e-30, 1e-33, 1e-36)])
def test_tiles_of_different_magnitudes(which, scales):
    """Each 32-row block, the unit of an exponent, at its own scale: V's exponent
    falls (O is rescaled) and rises, a zero tile sets none.  Scales that change
    inside a block are test_gpu_core_range.py's."""
    n = 160
    q, k, v, bias = _inputs(2, n, 5)
    s = torch.tensor(scales, device="cuda")[(torch.arange(n, device="cuda") // 32) % 3]
    t = {"q": q, "k": k, "v": v}[which]
    t.mul_(s[None, :, None, None] if which != "k" else s[None, :, None, None].clamp(max=30.0))
    _check(q, k, v, bias)


@pytest.mark.parametrize("gain", [30.0, 1e4, 3e7, 1e9])
def test_wide_logits_move_the_reference(gain):
    """Logits that rise from tile to tile, past 2^22 in log2 units too."""
    n = 132
    q, k, v, bias = _inputs(2, n, 9)
    bias = bias * gain + gain * torch.arange(n, device="cuda") / 16.0
    _check(q, k, v, bias)


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("which", ["q", "k", "v", "bias"])
@pytest.mark.parametrize("key", [3, 70, 99])
def test_non_finite_inputs_as_torch(which, value, key):
    n = 100
    q, k, v, bias = _inputs(2, n, 11)
    if which == "bias":
        bias[1, 5, key] = value
    else:
        {"q": q, "k": k, "v": v}[which][0, key, 2, 7] = value
    out, ref = _run(q, k, v, bias), _torch(q, k, v, bias, None, torch.float32)
    torch.testing.assert_close(out, ref, atol=2e-5, rtol=2e-5, equal_nan=True)


def test_bias_rows_beyond_32_bit_offsets():
    n, row = 4, (1 << 25) + 4
    q, k, v, bias = _inputs(2, n, 13)
    rows = torch.empty(4 * n, row, device="cuda")
    rows[:, :n] = bias.view(4 * n, n)
    out = _run(q, k, v, rows, row=row)
    torch.testing.assert_close(out, _torch(q, k, v, bias, None, torch.float32), atol=2e-6, rtol=0)


def test_non_finite_inputs_cost_no_more_than_fp32_products():
    """A batch whose every row holds a NaN runs on the FP32 matrix cores (2.2
    times the finite time here), not key by key (19 times).  Five times leaves
    room for noise on either side."""
    q, k, v, bias = _inputs(64, 512, 17)

    def seconds():
        for _ in range(2):
            _run(q, k, v, bias)
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        start.record()
        for _ in range(10):
            _run(q, k, v, bias)
        end.record()
        torch.cuda.synchronize()
        return start.elapsed_time(end)

    finite = min(seconds() for _ in range(3))
    k[:, 300, 1, 5] = float("nan")
    k[:, 300, 2, 5] = float("inf")
    v[:, 300, 0::3, 5] = float("nan")
    broken = min(seconds() for _ in range(3))
    print(f"finite {finite:.3f} ms, non-finite {broken:.3f} ms", flush=True)
    assert broken <= 5.0 * finite, (broken, finite)


@pytest.mark.parametrize("masked", [False, True])
def test_values_near_the_largest_float(masked):
    """A weighted mean of representable values is representable: nothing on the
    way to it (the sum before its division) may overflow."""
    n = 100
    q, k, v, bias = _inputs(2, n, 19)
    v *= 3e38 / v.abs().max()
    mask = torch.full((2, n), -3.0, device="cuda") if masked else None
    out = _run(q, k, v, bias, mask)
    assert torch.isfinite(out).all()
    ref = _torch(q, k, v, bias, mask, torch.float64)
    assert ((out.double() - ref).abs().max() / ref.abs().max()).item() <= 2e-6


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("gain", [1.0, 1e6, 3e10, 1e30])
def test_rows_without_an_unmasked_key_at_any_logit_size(gain, wide):
    """The logits of a fully masked row keep their distances at any size: from
    3e10 on, log2(e) times the largest is rounded by more than an exponential
    can hold.  wide: on the FP32 matrix cores too."""
    n = 100
    q, k, v, bias = _inputs(2, n, 20)
    bias = bias * gain
    if wide:
        v[:, 70] *= 1e9
        bias[:, :, 70] -= 1e4 * gain
    mask = torch.full((2, n), -1e9, device="cuda")
    out = _run(q, k, v, bias, mask).double()
    # the native order in float32, the rest in float64
    s = torch.matmul(*(t.permute(0, 2, 1, 3).contiguous() if i == 0 else
                       t.permute(0, 2, 3, 1).contiguous() for i, t in enumerate((q, k))))
    x = ((s + mask[:, None, None, :]) + bias).double()
    ref = torch.matmul(torch.softmax(x, -1), v.double().permute(0, 2, 1, 3).contiguous())
    err = (out - ref.permute(0, 2, 1, 3)).abs().amax((1, 2, 3))
    # q k flips a logit of the grid of 64 only where it lies near a midpoint: the sum
    # with -1e9 rounds it away, and both sides add the same bias to the same number
    assert torch.isfinite(out).all()
    assert (err <= 2e-6 * ref.abs().amax((1, 2, 3))).all(), err
