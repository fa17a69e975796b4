"""Performance cases of the pair stack: what a Pairformer run asks of this package.

Every case is one call through a public entry point (``triangle_attention_block``,
``triangle_multiplication``, ``transition``, ``dispatch_triangle_attention``,
OpenFold3's ``AttentionDispatcher``, the C ABI attention entries) or one pair
stack of five of them, at pair sizes N from a small domain to a long complex.
``listed()`` names the fixed ones, ``draw()`` gives others of the same ranges.

A case is a dict of plain values:

  op        "block" | "trimul" | "transition" | "operator" | "openfold3" |
            "abi" | "stack"
  n         residues (pair size); batch: outer rows of an attention call
  valid     residues kept by the mask on both axes (n: no mask is passed)
  ending    ending node (block, openfold3); outgoing: direction (trimul)
  dtype     "f32" | "bf16" (block)
  bias_gain spread of the triangle bias: logits of trained models span tens
"""
from __future__ import annotations

import math

import torch

from fireprot_amd import _native
from fireprot_amd import block as fb
from fireprot_amd import openfold3 as of3
from fireprot_amd import transition as ft
from fireprot_amd import triangle_attention as ta
from fireprot_amd import triangle_multiplication as tm

C, H, D = 128, 4, 32
INF = 1e9
DEVICE = "cuda"


def listed():
    return [
        # one small protein (the repository's c1): a call is mostly launches
        dict(name="block_f32_start_n124", op="block", n=124, valid=124, ending=False,
             dtype="f32", bias_gain=1.0),
        # a domain padded to a bucket size, ending node read through strides
        dict(name="block_f32_end_n256_tail", op="block", n=256, valid=231, ending=True,
             dtype="f32", bias_gain=4.0),
        # an ordinary protein with padding (c2)
        dict(name="block_f32_start_n512_tail", op="block", n=512, valid=461, ending=False,
             dtype="f32", bias_gain=1.0),
        # the headline size with its 12% padding and wide bias (c4)
        dict(name="block_f32_end_n1536_tail", op="block", n=1536, valid=1352, ending=True,
             dtype="f32", bias_gain=8.0),
        # BF16 storage, a crop size
        dict(name="block_bf16_start_n384", op="block", n=384, valid=384, ending=False,
             dtype="bf16", bias_gain=1.0),
        # BF16 storage, a long complex (c5)
        dict(name="block_bf16_end_n2048", op="block", n=2048, valid=2048, ending=True,
             dtype="bf16", bias_gain=1.0),
        # triangle multiplication of a domain, with a pair mask
        dict(name="trimul_out_n256_tail", op="trimul", n=256, valid=231, outgoing=True),
        # and of a long protein (c3's size, no multiple of a tile), no mask
        dict(name="trimul_in_n1000", op="trimul", n=1000, valid=1000, outgoing=False),
        # the pair transition of a crop
        dict(name="transition_n384", op="transition", n=384),
        # the reference's own attention benchmark through its C entry: one
        # 512-row chunk of the 1536-residue model, no mask
        dict(name="abi_b512_n1536", op="abi", batch=512, n=1536, valid=1536, bias_gain=1.0),
        # OpenFold3's _attention, ending-node wire layout, padded crop
        dict(name="openfold3_end_n384_tail", op="openfold3", batch=384, n=384, valid=350,
             ending=True, bias_gain=4.0),
        # a whole pair stack (five in-place updates) on a small padded protein
        dict(name="stack_n160_tail", op="stack", n=160, valid=147),
    ]


def draw(rng):
    def size(lo, hi):
        return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))

    def kept(n):  # no mask, or a padded tail of up to a fifth
        return n if rng.random() < 0.4 else max(1, n - rng.randint(1, max(1, n // 5)))

    op = rng.choice(["block"] * 5 + ["trimul"] * 3 + ["transition"] * 2
                    + ["operator", "openfold3", "abi", "stack"])
    gain = rng.choice([1.0, 4.0, 8.0])
    if op == "block":
        dtype = rng.choice(["f32", "f32", "bf16"])
        n = size(48, 1536)
        return dict(op=op, n=n, valid=kept(n), ending=rng.random() < 0.5, dtype=dtype,
                    bias_gain=gain)
    if op == "trimul":
        n = size(48, 1536)
        return dict(op=op, n=n, valid=kept(n), outgoing=rng.random() < 0.5)
    if op == "transition":
        return dict(op=op, n=size(48, 1536))
    if op == "stack":
        n = size(48, 512)
        return dict(op=op, n=n, valid=kept(n))
    n = size(48, 1536)
    if op == "abi":
        n = 4 * max(12, n // 4)
    batch = n if rng.random() < 0.5 else min(n, rng.choice([64, 128, 256, 512]))
    case = dict(op=op, batch=batch, n=n, valid=n if op == "abi" else kept(n), bias_gain=gain)
    if op == "openfold3":
        case["ending"] = rng.random() < 0.5
    return case


# ------------------------------------------------------------------ inputs

def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device=DEVICE) * scale


def _linear(g, out, fan_in=C, gain=1.0):
    return _randn(g, out, fan_in, scale=gain / math.sqrt(fan_in))


def _norm(g):
    return 1.0 + _randn(g, C, scale=0.1), _randn(g, C, scale=0.1)


def _pair(g, n):
    """A pair representation: unit-scale rows about per-channel means."""
    z = _randn(g, n, n, C)
    return z.mul_(2.0).add_(_randn(g, C))


def _mask(n, valid):
    if valid == n:
        return None
    keep = (torch.arange(n, device=DEVICE) < valid).float()
    return keep[:, None] * keep[None, :]


def _block_tensors(g, gain):
    ln_w, ln_b = _norm(g)
    return dict(ln_w=ln_w, ln_b=ln_b, w_q=_linear(g, C), w_k=_linear(g, C), w_v=_linear(g, C),
                w_g=_linear(g, C), b_g=1.0 + _randn(g, C, scale=0.1),
                w_bias=_linear(g, H, gain=gain), w_o=_linear(g, C), b_o=_randn(g, C, scale=0.1))


def _trimul_tensors(g):
    in_w, in_b = _norm(g)
    out_w, out_b = _norm(g)
    names = ("w_a_p", "w_a_g", "w_b_p", "w_b_g", "w_z", "w_g")
    return dict(ln_in_w=in_w, ln_in_b=in_b, ln_out_w=out_w, ln_out_b=out_b,
                **{k: _linear(g, C) for k in names})


def _transition_tensors(g):
    ln_w, ln_b = _norm(g)
    return dict(ln_w=ln_w, ln_b=ln_b, w_a=_linear(g, 4 * C), w_b=_linear(g, 4 * C),
                w_o=_linear(g, C, 4 * C))


def _attention_inputs(g, case):
    """q (scaled), k, v [B, 4, N, 32] views of head-last memory; the mask bias
    [B, 1, 1, N] or None; the triangle bias [1, 4, N, N]."""
    b, n, valid = case["batch"], case["n"], case["valid"]
    q, k, v = (_randn(g, b, n, H, D).transpose(1, 2) for _ in range(3))
    q.div_(math.sqrt(D))
    bias = _randn(g, n, n, H, scale=case["bias_gain"])
    # the ending node's bias and mask are transposed views of head-last memory
    bias = bias.permute(2, 1, 0) if case.get("ending") else bias.permute(2, 0, 1)
    mask = None
    if valid < n:
        keep = _mask(n, valid)
        full = INF * (keep - 1.0)
        mask = (full.t() if case.get("ending") else full)[:b, None, None, :]
    return q, k, v, mask, bias.unsqueeze(0)


def _draws(case, seed):
    """The tensors of a case, from the seed alone (shared by prepare and exact)."""
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    op = case["op"]
    if op in ("operator", "openfold3", "abi"):
        t = dict(zip(("q", "k", "v", "mask", "bias"), _attention_inputs(g, case)))
        if op == "openfold3" and t["mask"] is None:
            t["mask"] = torch.zeros(case["batch"], 1, 1, case["n"], device=DEVICE)
        if op == "abi":  # the entry's bias rows (1552 floats at N = 1536)
            n = case["n"]
            row = 1552 if n == 1536 else n
            rows = torch.zeros(1, H, n, row, device=DEVICE)
            rows[..., :n] = t["bias"]
            t["bias_rows"] = rows
        return t
    t = dict(z=_pair(g, case["n"]))
    if op != "transition":
        t["mask"] = _mask(case["n"], case["valid"])
    if op == "block":
        t["block"] = _block_tensors(g, case["bias_gain"])
        if case["dtype"] == "bf16":
            t["z"] = t["z"].bfloat16()
            t["block"] = {k: w.bfloat16() for k, w in t["block"].items()}
    elif op == "trimul":
        t["trimul"] = _trimul_tensors(g)
    elif op == "transition":
        t["transition"] = _transition_tensors(g)
    else:
        t["out"], t["in"] = _trimul_tensors(g), _trimul_tensors(g)
        t["start"], t["end"] = _block_tensors(g, 1.0), _block_tensors(g, 1.0)
        t["transition"] = _transition_tensors(g)
    return t


def _bytes(size):
    return torch.empty(int(size), dtype=torch.uint8, device=DEVICE)


def _native_attention(q, k, v, biases, **_):
    raise RuntimeError("the HIP attention did not take this call")


def prepare(case, seed):
    t = _draws(case, seed)
    op, n = case["op"], case["n"]
    s = dict(case=case, **t)
    if op == "block":
        dtype = t["z"].dtype
        s["w"] = fb.BlockWeights.from_tensors(**t["block"], inf=INF, dtype=dtype)
        s["ws"] = _bytes(fb.workspace_bytes(n, dtype))
    elif op == "trimul":
        s["w"] = tm.TriMulWeights.from_tensors(**t["trimul"])
        s["ws"] = _bytes(tm.workspace_bytes(n))
    elif op == "transition":
        s["w"] = ft.TransitionWeights.from_tensors(**t["transition"])
        s["ws"] = _bytes(_native.library().fpx_transition_workspace_bytes(n, n, C, 4))
    elif op == "stack":
        s["w_out"] = tm.TriMulWeights.from_tensors(**t["out"])
        s["w_in"] = tm.TriMulWeights.from_tensors(**t["in"])
        s["w_start"] = fb.BlockWeights.from_tensors(**t["start"], inf=INF)
        s["w_end"] = fb.BlockWeights.from_tensors(**t["end"], inf=INF)
        s["w_tr"] = ft.TransitionWeights.from_tensors(**t["transition"])
        s["ws_mul"] = _bytes(tm.workspace_bytes(n))
        s["ws"] = _bytes(fb.workspace_bytes(n))
        s["ws_tr"] = _bytes(_native.library().fpx_transition_workspace_bytes(n, n, C, 4))
    elif op == "openfold3":
        s["dispatcher"] = of3.AttentionDispatcher(of3.StridedAttention())
    elif op == "operator":
        s["module"] = torch.nn.Module().eval()
        s["biases"] = [t["bias"]] if t["mask"] is None else [t["mask"], t["bias"]]
    return s


def run(s):
    case = s["case"]
    op = case["op"]
    with torch.inference_mode():
        if op == "block":
            return fb.triangle_attention_block(s["z"], s["mask"], s["w"], ending=case["ending"],
                                               workspace=s["ws"])
        if op == "trimul":
            return tm.triangle_multiplication(s["z"], s["mask"], s["w"],
                                              outgoing=case["outgoing"], workspace=s["ws"])
        if op == "transition":
            return ft.transition(s["z"], s["w"], workspace=s["ws"])
        if op == "stack":
            # the recycled pair representation enters; the stack updates it in place
            z = s["z"].clone()
            for w, outgoing in ((s["w_out"], True), (s["w_in"], False)):
                tm.triangle_multiplication(z, s["mask"], w, outgoing=outgoing, out=z,
                                           accumulate=True, workspace=s["ws_mul"])
            fb.pair_step_triangle_attention(z, s["mask"], s["w_start"], s["w_end"],
                                            workspace=s["ws"])
            return ft.pair_transition_residual(z, s["w_tr"], workspace=s["ws_tr"])
        if op == "openfold3":
            return s["dispatcher"](_native_attention, s["q"], s["k"], s["v"],
                                   [s["mask"], s["bias"]])
        if op == "operator":
            return ta.dispatch_triangle_attention(module=s["module"], q=s["q"], k=s["k"],
                                                  v=s["v"], biases=s["biases"],
                                                  native=_native_attention)
        # the reference's ctypes loader: raw pointers, [B, N, 4, 32] operands
        q, k, v, bias = s["q"], s["k"], s["v"], s["bias_rows"]
        out = torch.empty((case["batch"], case["n"], H, D), device=q.device, dtype=q.dtype)
        _native.check(_native.library().fpx_attn_core_masked(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), None, 0, bias.data_ptr(), bias.stride(2),
            out.data_ptr(), case["batch"], case["n"],
            torch.cuda.current_stream(q.device).cuda_stream), "fpx_attn_core_masked")
        return out


# -------------------------------------------------------------------- work

def work(case):
    n, op = case["n"], case["op"]
    pair = n * n * C * 4
    core = 4 * H * D * n * n
    block = n * core + 2 * n * n * (C * 4 * C + C * H + C * C)
    trimul = 2 * n * n * C * C * 6 + 2 * n ** 3 * C
    transition = 2 * n * n * 3 * C * 4 * C
    if op == "block":
        e = 1 if case["dtype"] == "f32" else 2
        return dict(bytes=2 * pair / e + 4 * n * n * (case["valid"] < n), flops=block)
    if op == "trimul":
        return dict(bytes=2 * pair + 4 * n * n * (case["valid"] < n), flops=trimul)
    if op == "transition":
        return dict(bytes=2 * pair + 4 * 3 * C * 4 * C, flops=transition)
    if op == "stack":
        return dict(bytes=2 * pair + 4 * n * n * (case["valid"] < n),
                    flops=2 * trimul + 2 * block + transition)
    b = case["batch"]
    return dict(bytes=4 * b * n * C * 4 + 4 * H * n * n, flops=b * core)


def tolerance(case):
    """About four times the distance from ``exact`` measured over the ranges:
    float32 paths 1.4e-7 .. 7.5e-7 (largest element 1e-5 of its scale); BF16
    blocks 3e-3 (2e-2) at a unit bias, 9e-3 (1e-1) at wider ones, where the
    rounding of a stored logit term moves the weights more."""
    if case["op"] == "block" and case["dtype"] == "bf16":
        return {"rel": 1.2e-2, "max": 0.08} if case["bias_gain"] <= 1 else {"rel": 3e-2, "max": 0.4}
    return {"rel": 3e-6, "max": 4e-5}


# ------------------------------------------------- the same in 64-bit torch

def _ln(x, w, b):
    return torch.nn.functional.layer_norm(x, (C,), w, b, 1e-5)


def _core64(q, k, v, mask, bias, rows):
    """softmax(q k^T + mask + bias) v of the given outer rows (all float64).
    Rows with no kept key carry mask biases of -1e9, where the path's float32
    logits tie on a grid of 64: their logits are rounded where it rounds them."""
    n = q.shape[2]
    out = torch.empty(len(rows), H, n, D, dtype=torch.float64, device=q.device)
    step = max(1, (1 << 28) // (H * n * n))
    for at in range(0, len(rows), step):
        sel = rows[at:at + step]
        a = torch.matmul(q[sel], k[sel].transpose(-1, -2).contiguous())
        if mask is None:
            a += bias
        else:
            m = mask[sel]
            dead = (m.amax(-1) <= -INF / 2).flatten()
            if bool(dead.any()):
                x = (a[dead].float() + m[dead].float()) + bias.float()
                a += m
                a += bias
                a[dead] = x.double()
            else:
                a += m
                a += bias
        out[at:at + step] = torch.matmul(torch.softmax(a, dim=-1), v[sel])
    return out


def _block64(z, mask, w, ending):
    w = {k: t.double() for k, t in w.items()}
    x = z.transpose(0, 1) if ending else z
    if mask is not None:
        mask = (mask.t() if ending else mask).double()
        mask = (INF * (mask - 1.0))[:, None, None, :]
    x = _ln(x, w["ln_w"], w["ln_b"])
    n = x.shape[0]
    bias = (x @ w["w_bias"].t()).permute(2, 0, 1).contiguous()
    dz = torch.empty_like(x)
    step = max(1, (1 << 28) // (4 * n * C))
    for at in range(0, n, step):
        xs = x[at:at + step]
        q, k, v = ((xs @ w[name].t()).view(-1, n, H, D).transpose(1, 2).contiguous()
                   for name in ("w_q", "w_k", "w_v"))
        rows = torch.arange(len(xs), device=z.device)
        o = _core64(q / math.sqrt(D), k, v, None if mask is None else mask[at:at + step], bias,
                    rows)
        o = o.transpose(1, 2).reshape(-1, n, C)
        dz[at:at + step] = (o * torch.sigmoid(xs @ w["w_g"].t() + w["b_g"])) @ w["w_o"].t() \
            + w["b_o"]
    return dz.transpose(0, 1).contiguous() if ending else dz


def _trimul64(z, mask, w, outgoing):
    w = {k: t.double() for k, t in w.items()}
    x = _ln(z, w["ln_in_w"], w["ln_in_b"])
    m = 1.0 if mask is None else mask.double()[..., None]

    def side(name):
        t = m * torch.sigmoid(x @ w[f"w_{name}_g"].t()) * (x @ w[f"w_{name}_p"].t())
        return t.permute(2, 0, 1) if outgoing else t.permute(2, 1, 0)

    a, b = side("a").contiguous(), side("b").permute(0, 2, 1).contiguous()
    x2 = torch.bmm(a, b).permute(1, 2, 0)
    del a, b
    x2 = _ln(x2, w["ln_out_w"], w["ln_out_b"]) @ w["w_z"].t()
    return torch.sigmoid(x @ w["w_g"].t()) * x2


def _transition64(z, w):
    w = {k: t.double() for k, t in w.items()}
    out = torch.empty_like(z)
    for at in range(0, len(z), 64):
        x = _ln(z[at:at + 64], w["ln_w"], w["ln_b"])
        h = torch.nn.functional.silu(x @ w["w_a"].t()) * (x @ w["w_b"].t())
        out[at:at + 64] = h @ w["w_o"].t()
    return out


def exact(case, seed):
    t = _draws(case, seed)
    op = case["op"]
    with torch.inference_mode():
        if op in ("operator", "openfold3", "abi"):
            mask = None if t["mask"] is None else t["mask"].double()
            q, k, v = (t[x].double().contiguous() for x in "qkv")
            o = _core64(q, k, v, mask, t["bias"][0].double().contiguous(),
                        torch.arange(case["batch"], device=q.device))
            return o if op == "openfold3" else o.transpose(1, 2).contiguous()
        z = t["z"].double()
        if op == "block":
            return _block64(z, t["mask"], t["block"], case["ending"])
        if op == "trimul":
            return _trimul64(z, t["mask"], t["trimul"], case["outgoing"])
        if op == "transition":
            return _transition64(z, t["transition"])
        z = z + _trimul64(z, t["mask"], t["out"], True)
        z = z + _trimul64(z, t["mask"], t["in"], False)
        z = z + _block64(z, t["mask"], t["start"], False)
        z = z + _block64(z, t["mask"], t["end"], True)
        return z + _transition64(z, t["transition"])
