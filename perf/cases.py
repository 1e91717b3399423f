"""The workloads this package's speed is measured on.

Every case goes through entry points that a program using the package calls:
``TCFPLinear`` and ``TCFPMLP`` (training passes, and evaluation with the
weight quantised in the call), and the operator layer (activations quantised
and multiplied with weight codes that a serving program laid out once; the
raw dual GEMMs on operands that are already FP8).

Kinds of case and the sizes they range over:

* ``serve``  -- bf16 activations of a few tokens (generation, one to some
  tens of rows) or of a whole prompt (up to some thousands, any number), cast
  to FP8 and multiplied with stored W_hi / W_lo codes; bf16 output for the
  per-tensor format, the block format's fp32.
* ``eval``   -- ``TCFPLinear`` without autograd: the weight's dual
  quantisation is part of the call, as the layer defines it.
* ``gemm``   -- the dual GEMM alone, in each of its three scale formats.
* ``linear`` -- forward and backward of one ``TCFPLinear`` with error
  feedback: output, input gradient, weight and bias gradients, EF buffer.
* ``mlp``    -- forward and backward of Linear -> GELU -> Linear with an MSE
  loss, as ``fuse_tcfp_mlp`` builds it.

The sizes are those of the repository's own benchmark (4096^3 GEMMs, the
1024 -> 4096 -> 1024 MLP at 8192 tokens, d_model 256 with FFN 1024 at 4096
tokens, the 4096 -> 16384 layer at 8192 tokens) or generic ones.
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn
import torch.nn.functional as F

from tcfp_amd import core, ef_state
from tcfp_amd import kernels as K
from tcfp_amd.nn import TCFPLinear, fuse_tcfp_mlp

_E4M3, _E5M2 = torch.float8_e4m3fn, torch.float8_e5m2
_MAX = {_E4M3: 448.0, _E5M2: 57344.0}
_DT = {"bf16": torch.bfloat16, "fp32": torch.float32}

# Multiplying a weight by this stands for the optimiser's step between two
# training passes: the weight has changed, so the layer feeds its error back
# and rewrites the EF buffer.
_DECAY = 1.0 - 1e-6


def _case(kind, tokens, d_in, d_out, dtype="bf16", scaling="tensor", block=0, name=None):
    c = {"kind": kind, "tokens": tokens, "d_in": d_in, "d_out": d_out, "dtype": dtype,
         "scaling": scaling, "block": block}
    return c if name is None else {"name": name, **c}


def listed():
    return [
        # one generated token through a 1024-wide projection: the smallest
        # call there is, latency and launches
        _case("serve", 1, 1024, 1024, name="serve-1"),
        # a batch of 16 sequences generating, through the wide layer of the
        # scale-up configuration: both weight codes are read, little else
        _case("serve", 16, 4096, 16384, scaling="block", block=64, name="serve-16-block"),
        # a prompt of 1000 tokens (no multiple of any tile)
        _case("serve", 1000, 4096, 4096, name="serve-1000"),
        # evaluating a model in training on a small batch
        _case("eval", 64, 4096, 4096, name="eval-64"),
        # the headline product: 4096^3, per-tensor scales, bf16 output
        _case("gemm", 4096, 4096, 4096, name="gemm-4096"),
        # the same in the block format (power-of-two exponents along K)
        _case("gemm", 4096, 4096, 4096, dtype="fp32", scaling="block", block=64,
              name="gemm-4096-block"),
        # and with fp32 multipliers per block, 448 / amax
        _case("gemm", 4096, 4096, 4096, scaling="block_fp32", block=128, name="gemm-4096-fp32s"),
        # a training pass of the MLP configuration's first layer, per tensor
        _case("linear", 8192, 1024, 4096, name="linear-8192"),
        # a short last batch (1000 tokens) of a middle-sized layer whose
        # sides are no multiples of the tiles
        _case("linear", 1000, 1040, 1552, name="linear-1000"),
        # a training pass of the small transformer's FFN, block format, fp32
        # activations
        _case("linear", 4096, 256, 1024, dtype="fp32", scaling="block", block=64,
              name="linear-4096-block"),
        # a training pass of the scale-up layer: the largest
        _case("linear", 8192, 4096, 16384, scaling="block", block=64, name="linear-8192-block"),
        # the MLP configuration, forward and backward
        _case("mlp", 8192, 1024, 4096, name="mlp-8192"),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _dim(rng, lo, hi, step):
    return max(step, int(round(_log(rng, lo, hi) / step)) * step)


def draw(rng):
    kind = rng.choice(["serve", "serve", "eval", "gemm", "gemm", "linear", "linear", "mlp"])
    dtype = rng.choice(["bf16", "bf16", "fp32"])
    scaling, block = "tensor", 0
    if kind != "mlp" and rng.random() < 0.5:
        scaling, block = "block", rng.choice([32, 64, 64, 128])
        if kind == "gemm" and rng.random() < 0.4:
            scaling = "block_fp32"
    # sides: multiples of 16 (per tensor), of the block (block scales)
    step = block or 16
    d_in = _dim(rng, 256, 4096, step)
    d_out = _dim(rng, 256, 4096 if kind == "mlp" else 8192, step)
    if kind == "serve":
        # half of them generate (1 to 64 rows), half take a prompt in
        tokens = int(round(_log(rng, 1, 64) if rng.random() < 0.5 else _log(rng, 64, 4096)))
    elif kind == "eval":
        tokens = int(round(_log(rng, 1, 1024)))
    elif kind == "gemm":
        # fp32 multipliers take row counts that are multiples of 4
        tokens = 4 * int(round(_log(rng, 64, 2048)))
    else:
        # whole batches mostly, now and then a short last one of any length
        if rng.random() < 0.75:
            tokens = 64 * int(round(_log(rng, 4, 128)))
        else:
            tokens = int(round(_log(rng, 200, 2048)))
    if kind == "serve" and scaling == "tensor":
        dtype = "bf16"
    return _case(kind, tokens, d_in, d_out, dtype, scaling, block)


# ---------------------------------------------------------------- the inputs


def _inputs(case, seed):
    """x, w, b, g (and ef, w2, b2, target for the kinds that have them) of a
    case, made on the GPU from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    m, k, n = case["tokens"], case["d_in"], case["d_out"]
    dt = _DT[case["dtype"]]

    def randn(*shape, scale=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=gen, device="cuda") * scale).to(dtype)

    def weight(rows, cols):  # Kaiming-uniform, as the layers initialise
        return (torch.rand(rows, cols, generator=gen, device="cuda") * 2 - 1) / cols**0.5

    kind = case["kind"]
    d = {"x": randn(m, k, dtype=dt if kind != "gemm" else torch.bfloat16)}
    d["w"] = randn(n, k) if kind == "gemm" else weight(n, k)
    if kind == "gemm":
        return d
    d["b"] = weight(n, k)[:, 0].contiguous()
    if kind == "mlp":
        d["w2"], d["b2"] = weight(k, n), weight(k, n)[:, 0].contiguous()
        d["target"] = randn(m, k)
    if kind == "linear":
        # an output gradient of an averaged loss: small, and not of one size
        # over the columns
        d["g"] = randn(m, n, scale=1.0 / m) * (0.25 + torch.rand(n, generator=gen, device="cuda"))
    if kind in ("linear", "eval", "mlp"):
        # the error buffer of a training under way: below the last kept bit
        for wn in ("w", "w2"):
            if wn in d:
                d["ef" if wn == "w" else "ef2"] = randn(
                    *d[wn].shape, scale=float(2.0**-13 / d[wn].shape[1] ** 0.5))
    return d


def _layer(case, w, b, ef):
    layer = TCFPLinear(w.shape[1], w.shape[0], use_tensor_cores=True,
                       scale_block_size=case["block"] or None, device="cuda")
    with torch.no_grad():
        layer.weight.copy_(w)
        layer.bias.copy_(b)
    ef_state.load_ef_state_dict(layer, {"": {
        "_buffers": {"": ef}, "_amax_ema": {}, "_delayed_amax": {}, "_residual_ratio": {},
        "_step_count": {}, "_ema_decay": 0.999}})
    return layer


def prepare(case, seed):
    d = _inputs(case, seed)
    kind, scaling, bs = case["kind"], case["scaling"], case["block"]
    if kind in ("serve", "gemm"):
        # a serving program quantises its weights once
        if scaling == "tensor":
            d["wq"] = K.dual_quantize_per_tensor(d["w"])
        else:
            fmt = "fp32" if scaling == "block_fp32" else "exponent"
            d["wq"] = K.fused_dual_quantize_fp8(d["w"], bs, scale_format=fmt)
        if kind == "gemm":
            if scaling == "tensor":
                d["xq"] = core.to_fp8_e4m3(d["x"])
            else:
                d["xq"] = K.block_quantize_fp8(d["x"], bs, scale_format=fmt)
        return {"case": case, **d}
    s = {"case": case, "x": d["x"]}
    if kind == "mlp":
        mlp = nn.Sequential(_layer(case, d["w"], d["b"], d["ef"]), nn.GELU(),
                            _layer(case, d["w2"], d["b2"], d["ef2"]))
        s["model"], s["target"] = fuse_tcfp_mlp(mlp), d["target"]
    else:
        s["model"] = _layer(case, d["w"], d["b"], d["ef"])
        if kind == "linear":
            s["g"] = d["g"]
    if kind != "eval":
        s["x"] = d["x"].requires_grad_(True)
    return s


# ------------------------------------------------------------------ one pass


def _product(case, s):
    out = _DT[case["dtype"]]
    if case["scaling"] == "tensor":
        (q, inv), (hi, lo, inv_hi, inv_lo) = s["xq"], s["wq"]
        return K.fused_dual_gemm_forward(q, hi, lo, inv, inv_hi, inv_lo, bias=s.get("b"),
                                         out_dtype=out)
    (q, e), (hi, lo, e_hi, e_lo) = s["xq"], s["wq"]
    return K.fused_block_scaled_dual_gemm_forward(q, hi, lo, e, e_hi, e_lo, case["block"],
                                                  bias=s.get("b"), out_dtype=out)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "gemm":
        return _product(case, s)
    if kind == "serve":
        if case["scaling"] == "tensor":
            s["xq"] = core.to_fp8_e4m3(s["x"])
        else:
            s["xq"] = K.block_quantize_fp8(s["x"], case["block"])
        return _product(case, s)
    model, x = s["model"], s["x"]
    if kind == "eval":
        with torch.no_grad():
            return model(x)
    x.grad = None
    model.zero_grad(set_to_none=True)
    with torch.no_grad():
        torch._foreach_mul_([p for p in model.parameters() if p.ndim == 2], _DECAY)
    out = model(x)
    if kind == "linear":
        out.backward(s["g"])
        ef = model._error_state.get_error("", model.weight)
        return {"out": out.detach(), "dx": x.grad, "dw": model.weight.grad,
                "db": model.bias.grad, "ef": ef}
    loss = F.mse_loss(out, s["target"])
    loss.backward()
    return {"out": out.detach(), "loss": loss.detach(), "dx": x.grad,
            "dw1": model[0].weight.grad, "db1": model[0].bias.grad,
            "dw2": model[2].weight.grad, "db2": model[2].bias.grad}


# -------------------------------------------------------- what a pass needs


def work(case):
    kind, m, k, n = case["kind"], case["tokens"], case["d_in"], case["d_out"]
    ob = xb = 2 if case["dtype"] == "bf16" else 4
    mkn = float(m) * k * n
    scales = {"tensor": 0.0, "block": 1.0, "block_fp32": 4.0}[case["scaling"]]
    per_val = scales / case["block"] if case["block"] else 0.0
    if kind == "gemm":
        return {"bytes": m * k * (1 + per_val) + 2 * n * k * (1 + per_val) + m * n * ob,
                "flops": 4 * mkn}
    if kind == "serve":
        return {"bytes": m * k * xb + 2 * n * k * (1 + per_val) + 4 * n + m * n * ob,
                "flops": 4 * mkn}
    if kind == "eval":  # W and EF read
        return {"bytes": m * k * xb + 8 * n * k + 4 * n + m * n * 4, "flops": 4 * mkn}
    # W (read, and rewritten by its step), EF read and rewritten, dW
    weight = 20 * n * k + 8 * n
    if kind == "linear":
        return {"bytes": m * k * 2 * xb + weight + 2 * m * n * 4, "flops": 10 * mkn}
    # x, dx, target, out, both weights; the hidden activation needs no memory
    # of its own
    return {"bytes": m * k * (2 * xb + 8) + 2 * weight, "flops": 20 * mkn}


def tolerance(case):
    # The FP8 matrix instructions sum a 64-wide block with a relative error of
    # about 1.5e-5, whatever the order of the blocks; a bf16 output rounds at
    # 2^-9.  Everything that is quantised here is quantised from the inputs
    # themselves, so codes are the same -- except in the MLP, whose hidden
    # activation and its gradients are quantised from products: a code at a
    # rounding boundary flips, a whole E4M3 / E5M2 step for that value, twice
    # over by the time dw1 and dx are formed (1.1e-2 and 1.3e-2 against the
    # 64-bit evaluation; the output 8e-4).
    if case["kind"] == "mlp":
        return {"rel": 3e-2, "max": 0.9}
    # (bf16 results: a raw product's and a serving call's output, and the
    # gradient of a bf16 input)
    if case["kind"] != "eval" and case["dtype"] == "bf16":
        return {"rel": 4e-3, "max": 1e-2}
    return {"rel": 6e-5, "max": 3e-3}


# ------------------------------------------------ the same in 64 bits, plainly
#
# Quantised values are whole steps of their format, so the quantisation is
# evaluated by its rules (each operation rounded in the type the rule names);
# the products and sums of the dequantised values are in 64 bits.


def _cast(t, dtype):
    """(codes, 1 / scale): scale = max / amax, in t's type."""
    top = _MAX[dtype]
    scale = (top / t.abs().max().clamp(min=1e-12)).float()
    return (t.float() * scale).clamp(-top, top).to(dtype), 1.0 / scale


def _cast_blocks(t, bs, dtype, fp32_scales=False):
    """(codes [m, nb, bs], multiplier [m, nb, 1]) per block along a row."""
    top = _MAX[dtype]
    blocks = t.float().reshape(t.shape[0], -1, bs)
    amax = blocks.abs().amax(-1, keepdim=True).clamp(min=1e-12)
    if fp32_scales:
        if t.dtype == torch.bfloat16:
            scale = (top / amax.to(t.dtype)).float()
        else:
            scale = top / amax
        return (blocks * scale).clamp(-top, top).to(dtype), 1.0 / scale
    e = torch.ceil(torch.log2((amax / top).double()).float()).clamp(min=-126)
    return (blocks * torch.exp2(-e)).clamp(-top, top).to(dtype), torch.exp2(e)


def _values(t, case, dtype):
    """What t's codes stand for, fp32 (as the rules form it) and 64-bit."""
    if case["scaling"] == "tensor":
        q, inv = _cast(t, dtype)
    else:
        q, inv = _cast_blocks(t, case["block"], dtype, case["scaling"] == "block_fp32")
    return (q.float() * inv).reshape(t.shape), (q.double() * inv.double()).reshape(t.shape)


def _weights(w, ef, case):
    """W_hi + W_lo in 64 bits, and the new error buffer."""
    v = w if ef is None else w + ef
    hi, hi64 = _values(v, case, _E4M3)
    lo, lo64 = _values(v - hi, case, _E4M3)
    new = w - (hi + lo) if case["scaling"] == "tensor" else (w - hi) - lo
    return hi64 + lo64, new


def _forward(x, w64, b, case):
    x32, x64 = _values(x, case, _E4M3)
    out = x64 @ w64.t()
    return (out if b is None else out + b.double()), x32, x64


def _backward(g, w64, x32, x64, case):
    g64 = g.double()
    gq = _values(g, case, _E5M2)[1]
    if case["scaling"] == "tensor" and g.shape[0] % 16 == 0:
        dw = gq.t() @ x64
    else:
        # block scales, and token counts that the FP8 product does not take:
        # the gradient itself with the dequantised activation
        dw = g64.t() @ x32.double()
    return gq @ w64, dw, g64.sum(0)


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("gemm", "serve", "eval"):
        w64 = _weights(d["w"], d.get("ef"), case)[0]
        return _forward(d["x"], w64, d.get("b"), case)[0]
    w = d["w"] * _DECAY
    w64, ef = _weights(w, d["ef"], case)
    h, x32, x64 = _forward(d["x"], w64, d["b"], case)
    if kind == "linear":
        dx, dw, db = _backward(d["g"], w64, x32, x64, case)
        return {"out": h, "dx": dx, "dw": dw, "db": db, "ef": ef}
    # the layers hand on fp32 and quantise that
    h = h.float()
    w264, _ = _weights(d["w2"] * _DECAY, d["ef2"], case)
    a = F.gelu(h)
    out, a32, a64 = _forward(a, w264, d["b2"], case)
    diff = out - d["target"].double()
    g2 = (2.0 * diff / diff.numel()).float()
    da, dw2, db2 = _backward(g2, w264, a32, a64, case)
    hd = h.double()
    slope = 0.5 * (1 + torch.erf(hd / 2**0.5)) + hd * torch.exp(-hd * hd / 2) / (2 * math.pi) ** 0.5
    g1 = (da * slope).float()
    dx, dw1, db1 = _backward(g1, w64, x32, x64, case)
    return {"out": out, "loss": diff.square().mean(), "dx": dx, "dw1": dw1, "db1": db1,
            "dw2": dw2, "db2": db2}
