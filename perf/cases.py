"""Performance cases of the FP8 linear path: the calls that a program training or evaluating with FP8 linears makes,
through the package's public entry points, from layers of 128 features to a whole decoder block.

Every case is a dict of plain values.  `kind` says which entry points it takes:

  linear      one FP8Linear: a training step (forward, backward, weight re-quantisation where scaling is delayed), or a
              forward pass of a layer in evaluation mode
  block       several FP8Linears of a decoder layer: weight re-quantisation, forward and backward of each
  chain       FP8Linears that hand fp8 activations to each other and get fp8 gradients back
  quantise    FP8Tensor construction: current or delayed scaling, with or without the transposed copy
  dequantise  convert_tensor_from_fp8
  tex         the four Transformer-Engine-shaped functions in the order in which nanotron's own fp8 modules call them

Shapes come from the benchmark configurations and the tests of this repository (Llama-7B and Llama-3-8B linears at 4096
tokens, [4096, 4096] quantisation, the layer sizes of the linear sweep); activations are ~N(0, 1), weights ~N(0, 0.02),
output gradients ~N(0, 1e-3), and quantised tensors have heavy tails and outliers.
"""
import math

import torch

from nanotron_amd import tex_shim as tex
from nanotron_amd.fp8 import DelayedScaling, DTypes, FP8Linear, FP8Parameter, FP8Tensor
from nanotron_amd.fp8.dtypes import DType
from nanotron_amd.fp8.optim import requantize_fp8_weights
from nanotron_amd.fp8.tensor import convert_tensor_from_fp8

DEVICE = torch.device("cuda", 0)
TORCH = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"fp32": 4, "fp16": 2, "bf16": 2}
FP8 = {"e4m3": DTypes.FP8E4M3, "e5m2": DTypes.FP8E5M2}

# (in_features, out_features) of the layers of a block case, as multiples of what the case says
BLOCKS = {
    # gate, up, down
    "mlp": lambda c: [(c["hidden"], c["inter"]), (c["hidden"], c["inter"]), (c["inter"], c["hidden"])],
    # fused QKV (grouped-query heads), O, gate, up, down
    "layer": lambda c: [(c["hidden"], c["qkv"]), (c["hidden"], c["hidden"]), (c["hidden"], c["inter"]),
                        (c["hidden"], c["inter"]), (c["inter"], c["hidden"])],
}


def listed():
    return [
        # the reference's defaults (fp32, bias, every tensor scaled from its own amax) at the size of its model test:
        # the smallest training step, where launches and host time count
        dict(name="linear step 128 fp32", kind="linear", tokens=128, fin=128, fout=128, dtype="fp32", out="fp32",
             bias=True, delayed=False, accumulate=False, train=True),
        # benchmark configuration 1: one layer's forward pass in evaluation mode
        dict(name="linear eval 2048x1024x1024", kind="linear", tokens=2048, fin=1024, fout=1024, dtype="bf16", out="bf16",
             bias=False, delayed=True, accumulate=False, train=False),
        # a few tokens through a full-size projection: validation prompts, token-by-token generation
        dict(name="linear eval 16 tokens", kind="linear", tokens=16, fin=4096, fout=6144, dtype="bf16", out="bf16",
             bias=False, delayed=True, accumulate=False, train=False),
        # a batch whose token count is a multiple of nothing (unpadded sequences), biased layer of ordinary size
        dict(name="linear step 1021 tokens", kind="linear", tokens=1021, fin=1024, fout=2304, dtype="bf16", out="bf16",
             bias=True, delayed=True, accumulate=False, train=True),
        # layer sizes that are multiples of nothing either
        dict(name="linear step odd sizes", kind="linear", tokens=333, fin=515, fout=601, dtype="fp16", out="fp16",
             bias=False, delayed=True, accumulate=True, train=True),
        # benchmark configurations 3 and 4: the Llama-7B MLP, weight gradients accumulated in fp32
        dict(name="block llama-7b mlp", kind="block", layers="mlp", tokens=4096, hidden=4096, inter=11008, accumulate=True),
        # benchmark configuration 5, the headline: every linear of a Llama-3-8B decoder layer
        dict(name="block llama-3-8b layer", kind="block", layers="layer", tokens=4096, hidden=4096, qkv=6144, inter=14336,
             accumulate=False),
        # fp8 activations forward and fp8 gradients backward between three layers
        dict(name="chain 2048 tokens", kind="chain", tokens=2048, fin=1024, hidden=4096, fout=1024, dtype="bf16"),
        # benchmark configuration 2: both formats of one activation-sized tensor under delayed scaling
        dict(name="quantise 4096x4096 delayed", kind="quantise", rows=4096, cols=4096, dtype="bf16", formats="both",
             delayed=True, transpose=False),
        # an fp32 master weight with the transposed copy, scaled from its own amax
        dict(name="quantise weight transposed", kind="quantise", rows=11008, cols=4096, dtype="fp32", formats="e4m3",
             delayed=False, transpose=True),
        # back to high precision
        dict(name="dequantise 4096x4096", kind="dequantise", rows=4096, cols=4096, dtype="bf16", formats="e4m3"),
        # nanotron's own modules on the Transformer-Engine-shaped functions: casts, byte transposes, three GEMMs
        dict(name="tex linear 2048", kind="tex", tokens=2048, fin=2048, fout=2048, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi, grid):
    """A size between lo and hi, spread over its logarithm, on a grid of 256, 16 or 1 (clipped to the range)."""
    v = int(_log(rng, lo, hi))
    return max(lo, min(hi, (v + grid // 2) // grid * grid)) if v >= grid else max(lo, v)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "block", "block", "chain", "quantise", "quantise", "dequantise", "tex"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if kind == "linear":
        train = rng.random() < 0.65
        delayed = rng.random() < 0.7
        c = dict(kind=kind, train=train, delayed=delayed, dtype=dtype, out=dtype if delayed else rng.choice(["fp32", dtype]),
                 bias=rng.random() < 0.4, accumulate=train and rng.random() < 0.4)
        shape = rng.choice(["aligned", "aligned", "ragged tokens", "ragged tokens", "odd"])
        if not train and rng.random() < 0.5:   # few tokens, full-size layer
            return dict(c, tokens=_size(rng, 1, 128, 1), fin=_size(rng, 1024, 14336, 256), fout=_size(rng, 1024, 14336, 256))
        if shape == "aligned":
            return dict(c, tokens=_size(rng, 128, 4096, 16), fin=_size(rng, 128, 4096, 16), fout=_size(rng, 128, 4096, 16))
        if shape == "ragged tokens":
            return dict(c, tokens=_size(rng, 100, 2048, 1), fin=_size(rng, 256, 2048, 16), fout=_size(rng, 256, 2560, 16))
        return dict(c, tokens=_size(rng, 16, 700, 1), fin=_size(rng, 16, 700, 1), fout=_size(rng, 16, 700, 1))
    if kind == "block":
        hidden = _size(rng, 1024, 4096, 256)
        c = dict(kind=kind, layers=rng.choice(["mlp", "layer"]), tokens=_size(rng, 512, 4096, rng.choice([16, 256])), hidden=hidden,
                 inter=_size(rng, 2 * hidden, int(3.5 * hidden), 256), accumulate=rng.random() < 0.5)
        if c["layers"] == "layer":
            c["qkv"] = rng.choice([hidden + hidden // 2, 3 * hidden]) // 16 * 16
            if c["qkv"] > 6144:
                c["qkv"] = 6144
        return c
    if kind == "chain":
        return dict(kind=kind, tokens=_size(rng, 256, 4096, 16), fin=_size(rng, 512, 2048, 16), hidden=_size(rng, 1024, 4096, 16),
                    fout=_size(rng, 512, 2048, 16), dtype=rng.choice(["bf16", "fp32"]))
    if kind == "quantise":
        grid = rng.choice([128, 16, 1])
        return dict(kind=kind, rows=_size(rng, 128, 8192, grid), cols=_size(rng, 128, 8192, grid), dtype=dtype,
                    formats=rng.choice(["e4m3", "e5m2", "both"]), delayed=rng.random() < 0.5, transpose=rng.random() < 0.4)
    if kind == "dequantise":
        grid = rng.choice([128, 16, 1])
        return dict(kind=kind, rows=_size(rng, 128, 8192, grid), cols=_size(rng, 128, 8192, grid), dtype=dtype,
                    formats=rng.choice(["e4m3", "e5m2"]))
    return dict(kind=kind, tokens=_size(rng, 128, 4096, 16), fin=_size(rng, 128, 4096, 16), fout=_size(rng, 128, 4096, 16), dtype=dtype)


# ------------------------------------------------------------------------------------------------ states
def _normal(g, shape, std, dtype):
    return (torch.randn(shape, generator=g, device=DEVICE) * std).to(dtype)


def _heavy_tailed(g, shape, dtype):
    """Student-t with three degrees of freedom, scaled by 0.5, 0.01 % of the entries replaced by +-(50 .. 500)."""
    chi2 = torch.zeros(shape, device=DEVICE)
    for _ in range(3):
        chi2 += torch.randn(shape, generator=g, device=DEVICE).square_()
    x = torch.randn(shape, generator=g, device=DEVICE).mul_(0.5).div_(chi2.div_(3.0).sqrt_().clamp_min_(1e-3))
    u = torch.rand(shape, generator=g, device=DEVICE)
    v = torch.rand(shape, generator=g, device=DEVICE).mul_(450.0).add_(50.0)
    x = torch.where(u < 1e-4, torch.where(u < 5e-5, v, -v), x)
    return x.to(dtype)


def _layer(g, fin, fout, dtype, **kw):
    lin = FP8Linear(fin, fout, kw.pop("bias", False), DEVICE, dtype=dtype, **kw)
    lin.weight = FP8Parameter(_normal(g, (fout, fin), 0.02, dtype), DTypes.FP8E4M3)
    if lin.bias is not None:
        lin.bias.data.copy_(_normal(g, (fout,), 0.02, dtype))
    return lin


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    s = dict(kind=case["kind"])
    if case["kind"] == "linear":
        dt = TORCH[case["dtype"]]
        lin = _layer(g, case["fin"], case["fout"], dt, bias=case["bias"], out_dtype=TORCH[case["out"]],
                     delayed_scaling=case["delayed"], accumulate_grad=case["accumulate"])
        x = _normal(g, (case["tokens"], case["fin"]), 1.0, dt)
        s.update(lin=lin, x=x, train=case["train"], requantise=case["delayed"])
        s["gy"] = _normal(g, (case["tokens"], case["fout"]), 1e-3, TORCH[case["out"]])
        if case["train"] or case["delayed"]:   # in the middle of a run: the layer has stepped before and holds its scales
            _linear_step(dict(s, x=x.clone().requires_grad_(True)))
        if case["train"]:
            x.requires_grad_(True)
        else:
            lin.eval()
    elif case["kind"] == "block":
        bf = torch.bfloat16
        s["lins"], s["x"], s["gy"] = [], [], []
        for fin, fout in BLOCKS[case["layers"]](case):
            s["lins"].append(_layer(g, fin, fout, bf, out_dtype=bf, delayed_scaling=True, accumulate_grad=case["accumulate"]))
            s["x"].append(_normal(g, (case["tokens"], fin), 1.0, bf).requires_grad_(True))
            s["gy"].append(_normal(g, (case["tokens"], fout), 1e-3, bf))
        _block_step(s)
    elif case["kind"] == "chain":
        dt = TORCH[case["dtype"]]
        dims = [case["fin"], case["hidden"], case["hidden"], case["fout"]]
        s["lins"] = [_layer(g, a, b, dt, out_dtype=DTypes.FP8E4M3 if i < 2 else dt, delayed_scaling=True)
                     for i, (a, b) in enumerate(zip(dims, dims[1:]))]
        s["x"] = _normal(g, (case["tokens"], case["fin"]), 1.0, dt).requires_grad_(True)
        s["gy"] = _normal(g, (case["tokens"], case["fout"]), 1e-3, dt)
        _chain_step(s)
    elif case["kind"] == "quantise":
        s["x"] = _heavy_tailed(g, (case["rows"], case["cols"]), TORCH[case["dtype"]])
        s["transpose"] = case["transpose"]
        s["formats"] = [FP8[f] for f in (("e4m3", "e5m2") if case["formats"] == "both" else (case["formats"],))]
        s["states"] = [DelayedScaling(f, 16, 0, DEVICE) if case["delayed"] else None for f in s["formats"]]
        if case["delayed"]:
            run(s)
    elif case["kind"] == "dequantise":
        s["q"] = FP8Tensor(_heavy_tailed(g, (case["rows"], case["cols"]), TORCH[case["dtype"]]), FP8[case["formats"]])
        s["dtype"] = TORCH[case["dtype"]]
    else:
        dt = TORCH[case["dtype"]]
        one = torch.ones(1, device=DEVICE)
        s["x"] = _normal(g, (case["tokens"], case["fin"]), 1.0, dt)
        s["gy"] = _normal(g, (case["tokens"], case["fout"]), 1e-3, dt)
        w = FP8Tensor(_normal(g, (case["fout"], case["fin"]), 0.02, dt), DTypes.FP8E4M3)
        s["w"], s["sw_inv"] = w.as_subclass(torch.Tensor), w.fp8_meta.inverse_scale.reshape(1)
        # scales as the reference's FP8Meta holds them after an amax of 8 (X) and 0.008 (dY)
        s["sx"], s["sg"] = one * 32.0, one * 2.0 ** 22
        s["sx_inv"], s["sg_inv"] = 1 / s["sx"], 1 / s["sg"]
        s["empty"] = torch.empty(0, device=DEVICE)
    torch.cuda.synchronize()   # what a program did before this call is done
    return s


# ------------------------------------------------------------------------------------------------ passes
def _scales(lins):
    return [r._buf for lin in lins if lin.scaling is not None for r in lin.scaling.values()]


def _weight_grad(lin):
    return lin.weight.grad if lin.weight.dtype == torch.float32 else lin.weight.main_grad


def _linear_step(s):
    lin, x = s["lin"], s["x"]
    if s["requantise"]:
        requantize_fp8_weights(lin)
    x.grad = None
    if lin.bias is not None:
        lin.bias.grad = None
    y = lin(x)
    y.backward(s["gy"])
    return [y.detach(), x.grad, _weight_grad(lin), None if lin.bias is None else lin.bias.grad] + _scales([lin])


def _block_step(s):
    requantize_fp8_weights(s["lins"])
    out = []
    for lin, x, gy in zip(s["lins"], s["x"], s["gy"]):
        x.grad = None
        y = lin(x)
        y.backward(gy)
        out += [y.detach(), x.grad, _weight_grad(lin)]
    return out + _scales(s["lins"])


def _chain_step(s):
    requantize_fp8_weights(s["lins"])
    x = s["x"]
    x.grad = None
    h = x
    for lin in s["lins"]:
        h = lin(h)
    h.backward(s["gy"])
    return [h.detach(), x.grad] + [_weight_grad(lin) for lin in s["lins"]] + _scales(s["lins"])


def _cast(x, scale, inv, otype):
    return tex.cast_to_fp8(x, scale, torch.empty(1, device=DEVICE), inv, otype)


def _gemm(a, a_inv, at, b, b_inv, bt, e):
    d = torch.empty(b.shape[0], a.shape[0], device=DEVICE)
    tex.te_gemm(a, a_inv, at, True, b, b_inv, bt, False, d, e, DType.kFloat32, e, e, DType.kFloat32, e, False, e, 0, False, False, 0)
    return d


def _tex_step(s):
    e4, e5, e = DType.kFloat8E4M3, DType.kFloat8E5M2, s["empty"]
    xq = _cast(s["x"], s["sx"], s["sx_inv"], e4)
    y = _gemm(s["w"], s["sw_inv"], e4, xq, s["sx_inv"], e4, e)                                  # Y = X . W^T
    gq = _cast(s["gy"], s["sg"], s["sg_inv"], e5)
    dx = _gemm(tex.fp8_transpose(s["w"], e4), s["sw_inv"], e4, gq, s["sg_inv"], e5, e)          # dX = dY . W
    dw = _gemm(tex.fp8_transpose(xq, e4), s["sx_inv"], e4, tex.fp8_transpose(gq, e5), s["sg_inv"], e5, e)   # dW = dY^T . X
    return [xq, gq, y, dx, dw]


def run(state):
    kind = state["kind"]
    if kind == "linear":
        if state["train"]:
            return _linear_step(state)
        with torch.no_grad():
            return [state["lin"](state["x"])]
    if kind == "block":
        return _block_step(state)
    if kind == "chain":
        return _chain_step(state)
    if kind == "quantise":
        out = []
        for fmt, role in zip(state["formats"], state["states"]):
            q = FP8Tensor(state["x"], fmt, state=role, with_transpose=state["transpose"])
            out += [q.as_subclass(torch.Tensor), q.fp8_meta.amax, q.fp8_meta.scale]
            if state["transpose"]:
                out.append(q.transposed().as_subclass(torch.Tensor))
            if role is not None:
                out.append(role._buf)
        return out
    if kind == "dequantise":
        return [convert_tensor_from_fp8(state["q"], state["q"].fp8_meta, state["dtype"])]
    return _tex_step(state)


# ------------------------------------------------------------------------------------------------ what a pass needs
def _linear_work(tokens, fin, fout, hp, out, train, requantise, accumulate=False):
    """Bytes and FLOPs of one layer: high-precision tensors in and out once, the fp8 weight, the fp32 weight gradient."""
    x, y, w = tokens * fin, tokens * fout, fin * fout
    b = hp * x + w + out * y
    if not train:
        return b, 2.0 * tokens * fin * fout
    b += out * y + hp * x + 4 * w * (2 if accumulate else 1)
    if requantise:
        b += hp * w
    return b, 6.0 * tokens * fin * fout


def work(case):
    k = case["kind"]
    if k == "linear":
        b, f = _linear_work(case["tokens"], case["fin"], case["fout"], BYTES[case["dtype"]], BYTES[case["out"]], case["train"],
                            case["delayed"], case["accumulate"])
    elif k == "block":
        per = [_linear_work(case["tokens"], i, o, 2, 2, True, True, case["accumulate"]) for i, o in BLOCKS[case["layers"]](case)]
        b, f = sum(p[0] for p in per), sum(p[1] for p in per)
    elif k == "chain":
        dims, hp, t = [case["fin"], case["hidden"], case["hidden"], case["fout"]], BYTES[case["dtype"]], case["tokens"]
        w = sum(i * o for i, o in zip(dims, dims[1:]))
        b, f = 2 * hp * t * (case["fin"] + case["fout"]) + (hp + 1 + 4) * w, 6.0 * t * w
    elif k == "quantise":
        n, nf = case["rows"] * case["cols"], 2 if case["formats"] == "both" else 1
        b, f = n * (BYTES[case["dtype"]] + nf * (2 if case["transpose"] else 1)), 0.0
    elif k == "dequantise":
        b, f = case["rows"] * case["cols"] * (1 + BYTES[case["dtype"]]), 0.0
    else:
        x, y, w, hp = case["tokens"] * case["fin"], case["tokens"] * case["fout"], case["fin"] * case["fout"], BYTES[case["dtype"]]
        b, f = (hp + 1) * x + (hp + 1) * y + w + 4 * (x + y + w), 6.0 * case["tokens"] * case["fin"] * case["fout"]
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    """Quantised bytes, scales and dequantised values are exact.  GEMM results were compared with a product in 64 bits
    rounded once to the output's type; four times the differences seen (2-norm, largest element):
    fp32 outputs 1.5e-5 and 1.3e-4 (the matrix core aligns products before it adds them), fp16 8e-5 and one step of
    2^-10, bf16 2.3e-4 and one step of 2^-7.  A chain rounds activations and gradients to fp8 between its layers, where
    a difference of 1e-5 turns some bytes over to the next code: 8e-3 and 0.165 seen."""
    k = case["kind"]
    if k in ("quantise", "dequantise"):
        return "exact"
    if k == "chain":
        return {"rel": 0.03, "max": 0.66}
    if k == "tex" or (k == "linear" and case["dtype"] == "fp32" and case["out"] == "fp32"):
        return {"rel": 6e-5, "max": 5e-4}
    if k == "linear" and "bf16" not in (case["dtype"], case["out"]):
        return {"rel": 3.2e-4, "max": 4e-3}
    return {"rel": 1e-3, "max": 0.032}
