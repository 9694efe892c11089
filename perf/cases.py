"""The calls that a user of this package makes, as measurable cases.

A case is a dict of plain values. Five kinds cover the package's paths:

* ``quant``  one quantizer call (registry quantizers and the legacy
  per-tensor one) on an activation or a weight;
* ``linear`` an inference linear: quantize the activation, multiply by a
  weight that was quantized once (registry flow: ``quant.fn`` then ``bmm.fn``);
* ``heads``  a head-batched, block-scaled product of operands that are in fp8
  already (the MLA-style product);
* ``legacy`` the per-tensor ``fp8_bmm_quant`` call of the legacy tuple API,
  fp16 bias and output;
* ``layer``  one training step of ``Float8BMMLinear``: forward and backward,
  returning the output and every gradient.

``exact`` restates each in plain torch: the quantizers' own fp32 arithmetic
(it fixes which fp8 codes are multiplied), then products in 64 bits.
"""
from __future__ import annotations

import math

import torch

from practice_cuda_amd.fp8_bmm import fp8_bmm_quant, fp8_quant
from practice_cuda_amd.modules import Float8BlockBMMLinearConfig, Float8BMMLinear
from practice_cuda_amd.registry import QuantResult, get_bmm, get_quant

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
E4M3 = torch.float8_e4m3fn
FP8_MAX = 448.0
EPS = 1e-12


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one token's hidden state before a projection: all latency
        {"name": "quant_token", "kind": "quant", "scheme": "group", "rows": 1, "cols": 7168, "dtype": "bf16"},
        # a prefill chunk's hidden states, 1x128 groups (the activation quantizer's configuration)
        {"name": "quant_prefill", "kind": "quant", "scheme": "group", "rows": 4096, "cols": 7168, "dtype": "bf16"},
        # an MLP up-projection weight [K, N] with one scale per column: the right operand of the
        # channel-scaled product, and the quantizer's default axis
        {"name": "quant_weight_columns", "kind": "quant", "scheme": "column", "rows": 4096, "cols": 14336,
         "dtype": "bf16"},
        # the legacy per-tensor quantizer on one of its test shapes (32 heads x 2048 tokens of 960)
        {"name": "quant_legacy", "kind": "quant", "scheme": "legacy", "rows": 65536, "cols": 960, "dtype": "fp16"},
        # decoding sixteen sequences through the MLP up-projection, block-scaled
        {"name": "linear_decode", "kind": "linear", "scheme": "block", "batch": 1, "m": 16, "k": 4096, "n": 14336,
         "layout": "k", "bias": False, "activation": "none"},
        # a ragged prefill chunk through the same projection, channel scales, bias and GELU
        {"name": "linear_ragged", "kind": "linear", "scheme": "channel", "batch": 1, "m": 777, "k": 4096, "n": 14336,
         "layout": "n", "bias": True, "activation": "gelu"},
        # sizes that are multiples of nothing, batched (the shapes a caller with padded-free data has)
        {"name": "linear_odd", "kind": "linear", "scheme": "block", "batch": 3, "m": 1001, "k": 1031, "n": 777,
         "layout": "n", "bias": False, "activation": "none"},
        # MLA prefill: 128 heads, 2048 tokens, K 128 -> N 512
        {"name": "heads_prefill", "kind": "heads", "batch": 128, "m": 2048, "k": 128, "n": 512},
        # the same product while decoding a batch of 64 sequences
        {"name": "heads_decode", "kind": "heads", "batch": 128, "m": 64, "k": 128, "n": 512},
        # an ordinary shape of the legacy per-tensor product's published set, with its fp16 bias
        {"name": "legacy_bmm", "kind": "legacy", "batch": 80, "m": 2048, "n": 960, "k": 640, "layout": "n",
         "bias": True},
        # fine-tuning at a small batch: one short step of a narrow layer with a bias
        {"name": "layer_small", "kind": "layer", "recipe": "block", "batch": 1, "m": 512, "k": 1024, "n": 4096,
         "bias": True},
        # one GPU's share of a sharded training step: the MLP up-projection over 8192 tokens
        {"name": "layer_large", "kind": "layer", "recipe": "block", "batch": 1, "m": 8192, "k": 4096, "n": 14336,
         "bias": False},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of step between lo and hi, spread over their logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["quant", "quant", "linear", "linear", "heads", "legacy", "layer"])
    if kind == "quant":
        scheme = rng.choice(["group", "tile", "row", "column", "tensor", "legacy"])
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        cols = _log(rng, 256, 16384, rng.choice([1, 8, 128, 128]))
        rows = _log(rng, 1, min(65536, 60_000_000 // cols))
        return {"kind": kind, "scheme": scheme, "rows": rows, "cols": cols, "dtype": dtype}
    if kind == "linear":
        odd = rng.random() < 0.3
        batch = rng.choice([1, 1, 1, 3, 8]) if not odd else rng.choice([1, 3])
        k = _log(rng, 256, 4096 if not odd else 1200, 1 if odd else 128)
        n = _log(rng, 256, 14336 if not odd else 1200, 1 if odd else 16)
        m = _log(rng, 1, max(1, min(4096 if not odd else 1200, int(6e10 / (batch * k * n)))))
        return {"kind": kind, "scheme": rng.choice(["block", "channel", "tensor"]), "batch": batch, "m": m, "k": k,
                "n": n, "layout": rng.choice(["k", "n"]), "bias": rng.random() < 0.3,
                "activation": rng.choice(["none", "none", "gelu"])}
    if kind == "heads":
        return {"kind": kind, "batch": _log(rng, 16, 128), "m": _log(rng, 1, 2048), "k": rng.choice([128, 256, 512]),
                "n": rng.choice([128, 256, 512])}
    if kind == "legacy":
        return {"kind": kind, "batch": rng.choice([16, 32, 80]), "m": rng.choice([512, 1024, 2048]),
                "n": 80 * rng.choice([1, 2, 8, 12, 16, 20]), "k": 160 * rng.choice([1, 4, 6, 8, 10]),
                "layout": rng.choice(["n", "k"]), "bias": rng.random() < 0.8}
    batch = rng.choice([1, 1, 2, 4])
    k = _log(rng, 512, 4096, 128)
    n = _log(rng, 512, 8192, 128)
    m = _log(rng, 64, 8192 // batch, rng.choice([1, 128]))
    return {"kind": kind, "recipe": rng.choice(["block", "block", "tensor"]), "batch": batch, "m": m, "k": k, "n": n,
            "bias": rng.random() < 0.5}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _activation(shape, g, dtype=torch.bfloat16):
    """N(0, 1) with 0.1 % of the entries scaled by 50."""
    x = torch.randn(shape, generator=g, device="cuda")
    x *= torch.where(torch.rand(shape, generator=g, device="cuda") < 1e-3, 50.0, 1.0)
    return x.to(dtype)


def _normal(shape, g, std, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)


def _inputs(case, seed):
    """The case's high-precision tensors (legacy: its fp8 operands)."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "quant":
        shape = (case["rows"], case["cols"])
        make = _activation if case["scheme"] in ("group", "legacy", "tensor") else (
            lambda s, gen, dt: _normal(s, gen, 0.02, dt))
        return {"x": make(shape, g, DTYPES[case["dtype"]])}
    if kind == "linear":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        d = {"x": _activation((b, m, k), g),
             "w": _normal((b, n, k) if case["layout"] == "k" else (b, k, n), g, 0.02), "bias": None}
        if case["bias"]:
            d["bias"] = _normal((b, 1, n), g, 0.1)
        return d
    if kind == "heads":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        return {"x": _normal((b, m, k), g, 1.0), "w": _normal((b, k, n), g, 1.0)}
    if kind == "legacy":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        d = {"x": _normal((b, m, k), g, 1.0, torch.float32).to(E4M3),
             "w": _normal((b, k, n) if case["layout"] == "n" else (b, n, k), g, 1.0, torch.float32).to(E4M3),
             "scale": torch.rand((), generator=g, device="cuda") * 0.02 + 0.01, "bias": None}
        if case["bias"]:
            d["bias"] = _normal((b, m, n), g, 1.0, torch.float16)
        return d
    b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
    d = {"x": _normal((b, m, k), g, 1.0), "w": _normal((b, n, k), g, 0.02), "dy": _normal((b, m, n), g, 1e-3),
         "bias": None}
    if case["bias"]:
        d["bias"] = _normal((b, n), g, 0.02)
    return d


_QUANT_KWARGS = {
    "group": ("hip_per_block_2d", {"block_m": 1, "block_n": 128}),
    "tile": ("hip_per_block_2d", {"block_m": 128, "block_n": 128}),
    "row": ("hip_per_channel", {"channel_axis": -2}),
    "column": ("hip_per_channel", {"channel_axis": -1}),
    "tensor": ("hip_per_tensor", {}),
}
# scheme of a linear -> (quantizer of x, quantizer of w, product)
_LINEAR = {
    "block": ("group", "tile", "hip_per_block_2d_a_k_b_"),
    "channel": ("row", "column", "hip_per_channel_a_k_b_"),
    "tensor": ("tensor", "tensor", "hip_per_tensor_a_k_b_"),
}


def _quantizer(scheme):
    name, kwargs = _QUANT_KWARGS[scheme]
    fn = get_quant(name).fn
    return lambda x: fn(x, fp8_dtype=E4M3, **kwargs)


def prepare(case, seed):
    kind = case["kind"]
    d = _inputs(case, seed)
    if kind == "quant":
        return {"kind": kind, "x": d["x"], "fn": None if case["scheme"] == "legacy" else _quantizer(case["scheme"])}
    if kind in ("linear", "heads"):
        scheme = case.get("scheme", "block")
        qx, qw, name = _LINEAR[scheme]
        bmm = get_bmm(name + case.get("layout", "n"))
        w = d["w"] if case.get("layout", "n") == "n" else d["w"].transpose(-2, -1)
        state = {"kind": kind, "scheme": scheme, "bmm": bmm, "weight": bmm.prepare_b(_quantizer(qw)(w))}
        if kind == "heads":
            state["a"] = bmm.prepare_a(_quantizer(qx)(d["x"]))
            return state
        bias = d["bias"]
        state.update(x=d["x"], quant=_quantizer(qx), activation=case["activation"],
                     bias=None if bias is None else bias.expand(-1, case["m"], -1))
        return state
    if kind == "legacy":
        w = d["w"] if case["layout"] == "n" else d["w"].transpose(-2, -1)
        return {"kind": kind, "a": d["x"], "b": w, "bias": d["bias"], "scale": d["scale"]}
    layer = Float8BMMLinear(case["batch"], case["k"], case["n"], bias=case["bias"], device="cuda",
                            dtype=torch.bfloat16, config=Float8BlockBMMLinearConfig(granularity=case["recipe"]))
    with torch.no_grad():
        layer.weight.copy_(d["w"])
        if case["bias"]:
            layer.bias.copy_(d["bias"])
    return {"kind": kind, "layer": layer, "x": d["x"].requires_grad_(), "dy": d["dy"]}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "quant":
        if state["fn"] is None:
            return list(fp8_quant(state["x"]))
        q = state["fn"](state["x"])
        return [q.tensor, q.dequant_scale]
    if kind == "linear":
        bmm = state["bmm"]
        a = bmm.prepare_a(state["quant"](state["x"]))
        return bmm.fn(a, state["weight"], out_dtype=torch.bfloat16, bias=state["bias"],
                      activation=state["activation"], **bmm.prepare_call_kwargs(a, state["weight"]))
    if kind == "heads":
        return state["bmm"].fn(state["a"], state["weight"], out_dtype=torch.bfloat16)
    if kind == "legacy":
        return fp8_bmm_quant(state["a"], state["b"], state["bias"], quant_scale=state["scale"],
                             out_dtype=torch.float16)
    layer, x = state["layer"], state["x"]
    y = layer(x)
    wanted = [x, layer.weight] + ([layer.bias] if layer.bias is not None else [])
    return [y.detach(), *torch.autograd.grad(y, wanted, state["dy"])]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "quant":
        rows, cols = case["rows"], case["cols"]
        scales = {"group": rows * -(-cols // 128), "tile": -(-rows // 128) * -(-cols // 128), "row": rows,
                  "column": cols, "tensor": 1, "legacy": 1}[case["scheme"]]
        size = 4 if case["dtype"] == "fp32" else 2
        return {"bytes": rows * cols * (size + 1) + 4 * scales, "flops": 0}
    b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
    flops = 2 * b * m * n * k
    if kind == "linear":
        # bf16 x in, fp8 weight in, bf16 y out, bias
        return {"bytes": b * (2 * m * k + k * n + 2 * m * n + (2 * n if case["bias"] else 0)), "flops": flops}
    if kind == "heads":
        scales = m * -(-k // 128) + -(-k // 128) * -(-n // 128)
        return {"bytes": b * (m * k + k * n + 2 * m * n + 4 * scales), "flops": flops}
    if kind == "legacy":
        return {"bytes": b * (m * k + k * n + (4 if case["bias"] else 2) * m * n), "flops": flops}
    # x, w, dy in; y, dx, dw out (bf16)
    return {"bytes": 2 * b * 2 * (m * k + n * k + m * n), "flops": 3 * flops}


# ---------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------
def _div(num, s):
    return torch.full_like(s, num) / s


def _fp8(x, qs):
    return (x.float() * qs).clamp(-FP8_MAX, FP8_MAX).to(E4M3)


def _blocks(x, bm, bn):
    """x [B, M, N] zero-padded and cut into [B, M/bm, bm, N/bn, bn]."""
    b, m, n = x.shape
    x = torch.nn.functional.pad(x, (0, -n % bn, 0, -m % bm))
    return x.reshape(b, x.shape[1] // bm, bm, x.shape[2] // bn, bn)


def _block_values(x, bm, bn):
    """fp64 values of x quantized in bm x bn blocks."""
    b, m, n = x.shape
    t = _blocks(x, bm, bn)
    qs = _div(FP8_MAX, t.float().abs().amax(dim=(2, 4), keepdim=True).clamp(min=EPS))
    v = _fp8(t, qs).double() * _div(1.0, qs).double()
    return v.reshape(b, t.shape[1] * bm, t.shape[3] * bn)[:, :m, :n].contiguous()


def _channel_values(x, axis):
    s = x.float().abs().amax(dim=axis, keepdim=True).clamp(min=EPS)
    return _fp8(x, _div(FP8_MAX, s)).double() * (s / FP8_MAX).double()


def _tensor_values(x):
    qs = torch.reciprocal(x.float().abs().amax().clamp(min=EPS)) * FP8_MAX
    return _fp8(x, qs).double() * torch.reciprocal(qs).double()


def _tensorwise_values(x):
    """The training layer's per-tensor form: the division in 64 bits, rounded once."""
    qs = (FP8_MAX / x.float().abs().amax().double().clamp(min=EPS)).float()
    return _fp8(x, qs).double() * torch.reciprocal(qs).double()


def _product(a, b):
    return torch.bmm(a.contiguous(), b.contiguous())


def exact(case, seed):
    kind = case["kind"]
    d = _inputs(case, seed)
    if kind == "quant":
        x = d["x"].double().abs()
        scheme = case["scheme"]
        if scheme in ("group", "tile"):
            amax = _blocks(x[None], 1 if scheme == "group" else 128, 128).amax(dim=(2, 4))[0]
        elif scheme == "row":
            amax = x.amax(dim=-1)
        elif scheme == "column":
            amax = x.amax(dim=-2)
        else:
            amax = x.amax()
        return [None, amax.clamp(min=EPS) / FP8_MAX]
    x = d["x"]
    if kind == "legacy":
        w = d["w"] if case["layout"] == "n" else d["w"].transpose(-2, -1)
        out = _product(x.double(), w.double()) * d["scale"].double()
        return out if d["bias"] is None else out + d["bias"].double()
    if kind in ("linear", "heads"):
        w = d["w"] if case.get("layout", "n") == "n" else d["w"].transpose(-2, -1)
        scheme = case.get("scheme", "block")
        if scheme == "block":
            out = _product(_block_values(x, 1, 128), _block_values(w, 128, 128))
        elif scheme == "channel":
            out = _product(_channel_values(x, -1), _channel_values(w, -2))
        else:
            out = _product(_tensor_values(x), _tensor_values(w))
        if d.get("bias") is not None:
            out = out + d["bias"].double()
        return torch.nn.functional.gelu(out) if case.get("activation") == "gelu" else out
    w, dy = d["w"], d["dy"]
    if case["recipe"] == "block":
        qw = _block_values(w, 128, 128)
        y = _product(_block_values(x, 1, 128), qw.transpose(-2, -1))
        dx = _product(_block_values(dy, 1, 128), qw)
        dw = _product(_block_values(dy, 128, 1).transpose(-2, -1), _block_values(x, 128, 1))
    else:
        qx, qw, qdy = _tensorwise_values(x), _tensorwise_values(w), _tensorwise_values(dy)
        y, dx, dw = (_product(qx, qw.transpose(-2, -1)), _product(qdy, qw),
                     _product(qdy.transpose(-2, -1), qx))
    if d["bias"] is None:
        return [y, dx, dw]
    return [y + d["bias"].double().unsqueeze(1), dx, dw, dy.double().sum(dim=1)]


def tolerance(case):
    """Quantizers give the same bytes. Products: one rounding of the output to
    bf16 (2^-9 relative at most, 1.7e-3 in the 2-norm against 64 bits) or fp16
    (2^-12); fp32 sums in another order move a few values to a neighbour."""
    if case["kind"] == "quant":
        return "exact"
    if case["kind"] == "legacy":
        return {"rel": 1e-3}
    return {"rel": 7e-3}
