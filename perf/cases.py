"""What a user of this framework has it do, as cases that can be timed.

Five kinds of work, each through the public entry points:

  tensor / channel / group   quantize_tensor and, for 16-bit inputs,
                             dequantize_tensor of the result (fp32 inputs are
                             quantized only: dequantize_tensor returns 16-bit
                             tensors)
  linear                     the forward of cuBladeW8A16LinearLayer: INT8
                             weights quantized once, 16- or 32-bit activations,
                             optional LLM.int8 outlier columns and bias
  mlp                        down(silu(gate(x)) * up(x)) after quantize_model
  gemm                       wmma_gemm on dense operands

``listed()`` holds the named cases, ``draw(rng)`` makes more of the same
ranges, ``prepare`` / ``run`` make and run one, ``work`` / ``tolerance`` /
``exact`` say what it costs, how far two correct results may differ, and what
the result is in 64 bits.
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn

from cublade_amd.bindings.hip.wmma import wmma_gemm
from cublade_amd.quantization import (cuBladeW8A16LinearLayer, dequantize_tensor, quantize_model,
                                      quantize_tensor)

DEV = "cuda"
DTYPES = {
    "fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16,
    "fp8": torch.float8_e4m3fn, "int8": torch.int8, "uint8": torch.uint8,
}
SIZE = {"fp32": 4, "fp16": 2, "bf16": 2, "fp8": 1, "int8": 1, "uint8": 1}
N_OUTLIERS = 6


def listed() -> list[dict]:
    return [
        # A decode step's activations (16 tokens) to FP8 and back: latency.
        dict(name="fp8_tokens", kind="tensor", shape="16x4096", dtype="bf16", store="fp8"),
        # A large heavy-tailed tensor, one scale: the headline benchmark's step.
        dict(name="int8_tensor", kind="tensor", shape="8192x8192", dtype="fp16", store="int8"),
        # An fp32 nn.Linear weight to INT8 rows: what quantize_model does to
        # every layer of a model that was never cast to 16 bits.
        dict(name="int8_rows_fp32", kind="channel", shape="11008x4096", dtype="fp32", axis=0),
        # The same weight in bf16 with one scale per input feature.
        dict(name="int8_cols", kind="channel", shape="11008x4096", dtype="bf16", axis=1),
        # Groups whose size is no multiple of a 16-byte load, odd row count.
        dict(name="int8_group_ragged", kind="group", shape="4099x1400", dtype="fp16", axis=1,
             group=100),
        # A large cache or activation tensor in groups of 128.
        dict(name="int8_group", kind="group", shape="16384x14336", dtype="bf16", axis=1,
             group=128),
        # Decode through an up projection: 16 tokens, outlier columns.
        dict(name="linear_decode", kind="linear", m=16, n=11008, k=4096, dtype="fp16",
             outliers=True, bias=False),
        # Decode through the matching down projection: few tokens, long rows.
        dict(name="linear_down", kind="linear", m=4, n=4096, k=11008, dtype="bf16",
             outliers=False, bias=True),
        # Prefill of 4096 tokens with outlier columns.
        dict(name="linear_prefill", kind="linear", m=4096, n=11008, k=4096, dtype="fp16",
             outliers=True, bias=False),
        # The layer of a model left in fp32: fp32 activations, a ragged batch.
        dict(name="linear_fp32", kind="linear", m=500, n=11008, k=4096, dtype="fp32",
             outliers=False, bias=True),
        # A whole MLP block after quantize_model, a short prompt.
        dict(name="mlp_block", kind="mlp", m=200, hidden=4096, inter=11008, dtype="bf16"),
        # The dense GEMM with B as [K, N].
        dict(name="gemm_int8", kind="gemm", m=2048, n=2048, k=2048, dtype="int8", layout="kn"),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _ragged(rng, v: int, step: int) -> int:
    """v as it is (one time in three), else rounded to a multiple of step."""
    return v if rng.random() < 1 / 3 else max(step, v // step * step)


def draw(rng) -> dict:
    kind = rng.choice(["tensor", "tensor", "channel", "channel", "channel", "group", "group",
                       "linear", "linear", "linear", "linear", "linear", "mlp", "gemm", "gemm"])
    if kind in ("tensor", "channel", "group"):
        store = rng.choice(["fp8", "int8"]) if kind == "tensor" else "int8"
        dtype = rng.choice(["fp16", "bf16"] if store == "fp8" else ["fp16", "bf16", "fp32"])
        rows, cols = _log_int(rng, 1, 8192), _ragged(rng, _log_int(rng, 64, 14336), 64)
        cols = min(cols, (1 << 26) // rows)
        if kind == "tensor":
            return dict(kind=kind, shape=f"{rows}x{cols}", dtype=dtype, store=store)
        if kind == "channel":
            if rng.random() < 0.25:   # a middle axis
                return dict(kind=kind, shape=f"{rng.randint(2, 8)}x{max(1, rows // 8)}x{cols}",
                            dtype=dtype, axis=1)
            return dict(kind=kind, shape=f"{rows}x{cols}", dtype=dtype, axis=rng.randint(0, 1))
        group = rng.choice([32, 64, 100, 128, 256])
        if rng.random() < 0.3:        # groups along the rows
            rows = max(1, rows // group) * group
            cols = min(cols, (1 << 26) // rows)
            return dict(kind=kind, shape=f"{rows}x{cols}", dtype=dtype, axis=0, group=group)
        return dict(kind=kind, shape=f"{rows}x{max(1, cols // group) * group}", dtype=dtype, axis=1,
                    group=group)
    if kind == "linear":
        dtype = rng.choice(["fp16", "fp16", "bf16", "bf16", "fp32"])
        n = _ragged(rng, _log_int(rng, 256, 14336), 64)
        step = rng.choice([64, 64, 64, 64, 16, 2])   # of the row length
        k = _log_int(rng, 256, 14336) // step * step
        # fp32 activations and rows off the 16-element grid take more time per product
        cap = (4096 if dtype != "fp32" else 700) * 11008 * 4096
        if k % 16:
            cap = 100 * 11008 * 4096
        m = _log_int(rng, 1, max(1, min(4096, cap // (n * k))))
        return dict(kind=kind, m=m, n=n, k=k, dtype=dtype,
                    outliers=dtype != "fp32" and rng.random() < 0.4, bias=rng.random() < 0.5)
    if kind == "mlp":
        hidden = rng.choice([1024, 2048, 4096])
        return dict(kind=kind, m=_log_int(rng, 1, 1024), hidden=hidden,
                    inter=_log_int(rng, 2 * hidden, min(4 * hidden, 11008)) // 64 * 64,
                    dtype=rng.choice(["fp16", "bf16"]))
    m, n, k = (_log_int(rng, 256, 4096) // 16 * 16 for _ in range(3))
    return dict(kind=kind, m=m, n=n, k=k, dtype=rng.choice(["int8", "uint8", "fp16", "bf16"]),
                layout=rng.choice(["kn", "nk"]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _shape(case: dict) -> tuple[int, ...]:
    return tuple(int(d) for d in case["shape"].split("x"))


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _quant_input(case: dict, seed: int) -> torch.Tensor:
    """Heavy-tailed for one scale per tensor (0.5 x Student-t, 3 degrees of
    freedom), a weight's N(0, 0.02) with a few large columns for channels,
    N(0, 1) with a factor per row for groups."""
    g, shape = _gen(seed), _shape(case)
    x = torch.randn(shape, generator=g, device=DEV)
    if case["kind"] == "tensor":
        d = torch.randn(shape, generator=g, device=DEV).square_()
        for _ in range(2):
            d += torch.randn(shape, generator=g, device=DEV).square_()
        x.mul_(0.5).mul_(d.div_(3).rsqrt_()).clamp_(-6e4, 6e4)
    elif case["kind"] == "channel":
        x.mul_(0.02)
        big = torch.randint(0, shape[-1], (max(1, shape[-1] // 1000),), generator=g, device=DEV)
        x[..., big] *= 20
    else:
        x.mul_(0.1 + 9.9 * torch.rand((shape[0],) + (1,) * (len(shape) - 1), generator=g,
                                      device=DEV))
    return x.to(DTYPES[case["dtype"]])


def _linear_inputs(case: dict, seed: int):
    """(x, weight, bias or None, outlier columns): x ~ N(0, 1) with a few
    feature columns at +-U(8, 20) where the case has outliers."""
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    m, n, k = case["m"], case["n"], case["k"]
    x = torch.randn(m, k, generator=g, device=DEV)
    cols = torch.empty(0, dtype=torch.long, device=DEV)
    if case["outliers"]:
        cols = torch.sort(torch.randperm(k, generator=g, device=DEV)[:N_OUTLIERS]).values
        x.clamp_(-5.5, 5.5)
        mag = 8 + 12 * torch.rand(m, N_OUTLIERS, generator=g, device=DEV)
        x[:, cols] = torch.sign(torch.randn(m, N_OUTLIERS, generator=g, device=DEV)) * mag
    w = 0.02 * torch.randn(n, k, generator=g, device=DEV)
    b = 0.1 * torch.randn(n, generator=g, device=DEV) if case["bias"] else None
    return x.to(dt), w.to(dt), None if b is None else b.to(dt), cols


class Mlp(nn.Module):
    def __init__(self, hidden: int, inter: int, dtype: torch.dtype):
        super().__init__()
        kw = dict(bias=False, device=DEV, dtype=dtype)
        self.gate_proj = nn.Linear(hidden, inter, **kw)
        self.up_proj = nn.Linear(hidden, inter, **kw)
        self.down_proj = nn.Linear(inter, hidden, **kw)

    def forward(self, x):
        return self.down_proj(torch.nn.functional.silu(self.gate_proj(x)) * self.up_proj(x))


def _mlp_inputs(case: dict, seed: int):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    h, i = case["hidden"], case["inter"]
    x = torch.randn(case["m"], h, generator=g, device=DEV).to(dt)
    ws = [(0.02 * torch.randn(s, generator=g, device=DEV)).to(dt) for s in ((i, h), (i, h), (h, i))]
    return x, ws


def _gemm_inputs(case: dict, seed: int):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    m, n, k = case["m"], case["n"], case["k"]
    b_shape = (k, n) if case["layout"] == "kn" else (n, k)

    def make(shape):
        if case["dtype"] in ("fp16", "bf16"):
            return torch.randn(shape, generator=g, device=DEV).to(dt)
        lo = 0 if case["dtype"] == "uint8" else -128
        return torch.randint(lo, lo + 256, shape, generator=g, device=DEV, dtype=torch.int16).to(dt)

    a, b = make((m, k)), make(b_shape)
    return a, b if case["layout"] == "kn" else b.t()


def prepare(case: dict, seed: int):
    """What the program holds before the call: the input tensor, the
    quantized layer or block with its activations, or the GEMM's operands."""
    kind = case["kind"]
    if kind in ("tensor", "channel", "group"):
        kw = dict(dtype=DTYPES[case.get("store", "int8")], mode=kind)
        if kind != "tensor":
            kw["ch_axis"] = case["axis"]
        if kind == "group":
            kw["group_size"] = case["group"]
        return dict(kind="quant", x=_quant_input(case, seed), kw=kw)
    if kind == "linear":
        x, w, b, _ = _linear_inputs(case, seed)
        layer = cuBladeW8A16LinearLayer(case["k"], case["n"], bias=b is not None, dtype=w.dtype,
                                        handle_outliers=case["outliers"],
                                        outlier_mode="activation" if case["outliers"] else "weight")
        layer.quantize(w, x if case["outliers"] else None)
        if b is not None:
            layer.bias = nn.Parameter(b, requires_grad=False)
        return dict(kind="module", module=layer, x=x)
    if kind == "mlp":
        x, ws = _mlp_inputs(case, seed)
        block = Mlp(case["hidden"], case["inter"], x.dtype).eval()
        with torch.no_grad():
            for p, w in zip(block.parameters(), ws):
                p.copy_(w)
        return dict(kind="module", module=quantize_model(block, "w8a16"), x=x)
    a, b = _gemm_inputs(case, seed)
    return dict(kind="gemm", a=a, b=b)


def run(state):
    if state["kind"] == "quant":
        qt = quantize_tensor(state["x"], **state["kw"])
        if qt.original_dtype == torch.float32:
            return qt.data, qt.scale
        return qt.data, qt.scale, dequantize_tensor(qt)
    if state["kind"] == "module":
        with torch.no_grad():
            return state["module"](state["x"])
    return wmma_gemm(state["a"], state["b"])


# ---------------------------------------------------------------------------
# Cost, tolerance, the result in 64 bits
# ---------------------------------------------------------------------------
def _scales(case: dict) -> int:
    shape = _shape(case)
    if case["kind"] == "tensor":
        return 1
    if case["kind"] == "channel":
        return shape[case["axis"]]
    return math.prod(shape) // case["group"]


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("tensor", "channel", "group"):
        n, e, s = math.prod(_shape(case)), SIZE[case["dtype"]], 4 * _scales(case)
        quant = n * e + n + s
        return {"bytes": quant + (0 if e == 4 else n + s + n * e), "flops": 0}
    if kind == "linear":
        m, n, k, e = case["m"], case["n"], case["k"], SIZE[case["dtype"]]
        out = N_OUTLIERS if case["outliers"] else 0
        return {"bytes": n * k + e * (m * k + m * n + n * (1 + case["bias"] + out)) + 8 * out,
                "flops": 2 * m * n * (k + out)}
    if kind == "mlp":
        m, h, i = case["m"], case["hidden"], case["inter"]
        return {"bytes": 3 * h * i + 2 * (2 * i + h) + 2 * 2 * m * h, "flops": 3 * 2 * m * h * i}
    m, n, k, e = case["m"], case["n"], case["k"], SIZE[case["dtype"]]
    return {"bytes": e * (m * k + k * n) + 4 * m * n, "flops": 2 * m * n * k}


def tolerance(case: dict):
    """Codes, scales and dequantized values are defined to the bit, integer
    products too. Floating-point sums: about four times the distance of
    the path from ``exact`` over these ranges. fp32 activations keep 16
    significant bits on the matrix cores (rows that are a multiple of 64)."""
    kind, dt = case["kind"], case["dtype"]
    if kind in ("tensor", "channel", "group") or dt in ("int8", "uint8"):
        return "exact"
    if kind == "gemm":                       # fp32 result of exact 16-bit products
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "mlp":
        return {"rel": 1.6e-2 if dt == "bf16" else 2e-3}
    if dt == "fp32":
        return {"rel": 2e-5, "max": 1.2e-4} if case["k"] % 64 == 0 else {"rel": 2e-6, "max": 1e-5}
    return {"rel": 6.7e-3, "max": 1.6e-2} if dt == "bf16" else {"rel": 8.3e-4, "max": 2e-3}


def _int8_rows(w: torch.Tensor):
    """INT8 codes and fp32 scales of a weight, one scale per row."""
    amax = w.float().abs().amax(dim=1, keepdim=True).clamp_min(1e-12)
    inv = torch.full_like(amax, 127.0) / amax   # one rounding (a scalar over a tensor takes two)
    return torch.round(w.float() * inv).clamp_(-127, 127), (1.0 / inv).squeeze(1)


def _linear64(x, w, b, cols):
    keep = w
    if cols.numel():
        keep = w.clone()
        keep[:, cols] = 0
    codes, scale = _int8_rows(keep)
    y = (x.double() @ codes.double().t()) * scale.to(w.dtype).double()
    if cols.numel():
        y += x[:, cols].double() @ w[:, cols].double().t()
    return y if b is None else y + b.double()


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("tensor", "channel", "group"):
        x, shape = _quant_input(case, seed).double(), _shape(case)
        if kind == "tensor":
            amax = x.abs().amax()
            s, scale = amax, amax
        elif kind == "channel":
            dims = [d for d in range(len(shape)) if d != case["axis"]]
            s = x.abs().amax(dim=dims, keepdim=True)
            scale = s.flatten()
        elif case["axis"] == 1:
            grouped = x.view(shape[0], -1, case["group"]).abs().amax(dim=2)
            s, scale = grouped.repeat_interleave(case["group"], dim=1), grouped.flatten()
        else:
            grouped = x.view(-1, case["group"], shape[1]).abs().amax(dim=1)
            s, scale = grouped.repeat_interleave(case["group"], dim=0), grouped.t().flatten()
        if case.get("store") == "fp8":
            codes = (x * (448 / s.clamp_min(1e-12))).clamp_(-448, 448).to(torch.float8_e4m3fn)
            return codes, scale / 448, codes.double() * (s / 448)
        codes = torch.round(x * (127 / s.clamp_min(1e-12))).clamp_(-127, 127)
        if case["dtype"] == "fp32":
            return codes, scale / 127
        return codes, scale / 127, codes * (s / 127)
    if kind == "linear":
        return _linear64(*_linear_inputs(case, seed))
    if kind == "mlp":
        x, (wg, wu, wd) = _mlp_inputs(case, seed)
        none = torch.empty(0, dtype=torch.long, device=DEV)
        gate, up = _linear64(x, wg, None, none), _linear64(x, wu, None, none)
        return _linear64(torch.nn.functional.silu(gate) * up, wd, None, none)
    a, b = _gemm_inputs(case, seed)
    y = a.double() @ b.double()
    return y if case["dtype"] in ("fp16", "bf16") else y.to(torch.int64)
