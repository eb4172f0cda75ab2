"""The measured workloads of the W8A8 linears: what a diffusion-transformer user has the library do, through its public
entry points, from one-row calls to the linears of a 720p video.

A case is one pass of one of three things a program does:

  linear    the forward of a converted ``nn.Linear`` (bf16 / fp16 / fp32 in and out); ``scheme`` says how it was converted:
            "token"   dynamic per-token activations, per-channel weights (``quantize_dynamic``, the DiT's scheme)
            "tensor"  dynamic per-tensor activations and weights (the library's default dynamic configuration)
            "static"  calibrated per-tensor activation scale, per-channel weights (``prepare`` / ``convert``)
  ffn       LayerNorm + modulation + quantisation -> up projection -> GELU + quantisation -> down projection: the
            feed-forward of a block whose producers are fused (``fuse_transformer_blocks``)
  convert   the conversion of a float linear: statistics, scales and bytes of its weight (``Linear.from_float``)

Inputs follow bench.py's recipe: activations are normal with 1 % of the channels twenty times larger, weights 0.02
times normal, biases 0.01 times normal.
"""
import math

import torch
from torch import nn

from dax_amd.adapters.wan.block_fusion import gelu_tanh_quant, layernorm_quant
from dax_amd.quant.nn.dynamic import Linear
from dax_amd.quant.quantization import convert, prepare as prepare_static, quantize_dynamic
from dax_amd.quant.quantization.qconfig import (
    get_default_dynamic_fp8_qconfig,
    get_default_dynamic_int8_qconfig,
    get_dynamic_fp8_per_token_act_per_channel_weight_qconfig,
    get_dynamic_int8_per_token_act_per_channel_weight_qconfig,
    get_fp8_per_channel_weight_qconfig,
)

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}
ACT = {"int8": torch.int8, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
DEV = "cuda"
LN_EPS = 1e-6
LARGEST = 75600 * 5120 * 13824  # multiply-adds of the largest listed case


def _linear(name, m, k, n, fmt="int8", scheme="token", dtype="bf16", bias=True):
    case = {"kind": "linear", "m": m, "k": k, "n": n, "fmt": fmt, "scheme": scheme, "dtype": dtype, "bias": bias}
    return dict(case, name=name) if name else case


def _ffn(name, m, k, n, fmt):
    case = {"kind": "ffn", "m": m, "k": k, "n": n, "fmt": fmt}
    return dict(case, name=name) if name else case


def _convert(name, n, k, fmt, dtype="bf16"):
    case = {"kind": "convert", "n": n, "k": k, "fmt": fmt, "dtype": dtype}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one row: a conditioning vector (time step, pooled prompt) through a 1536-wide projection; the smallest call
        _linear("row_int8", 1, 1536, 1536),
        # a handful of rows against a 5120-wide weight: short prompts, registers, a few conditioning tokens
        _linear("rows17_e4m3", 17, 5120, 5120, "e4m3"),
        # the 512 text tokens of cross-attention's k / v projections
        _linear("text512_int8", 512, 5120, 5120),
        # the single linear that the CPU path is quoted on: a small latent, every channel dimension 1536
        _linear("tokens4096_int8", 4096, 1536, 1536),
        # an fp16 module with channel counts that are multiples of nothing much (adapters, control branches, pruned widths)
        _linear("ragged2900_fp16", 2900, 1000, 3080, dtype="fp16"),
        # the library's default dynamic FP8 configuration: per-tensor scales, e5m2 activations
        _linear("tensor4096_e5m2", 4096, 5120, 5120, "e5m2", "tensor"),
        # a calibrated static FP8 module at one micro-batch of an eight-way sequence-parallel rank
        _linear("static4725_e4m3", 4725, 5120, 5120, "e4m3", "static"),
        # the feed-forward of a fused block at the rows one of eight sequence-parallel ranks holds
        _ffn("ffn9450_e4m3", 9450, 5120, 13824, "e4m3"),
        # QKV of the 1.3B model at 480p: many rows, short K
        _linear("video480p_qkv_int8", 32760, 1536, 4608),
        # the out-projection of the 14B model at 720p, FP8
        _linear("video720p_out_e4m3", 75600, 5120, 5120, "e4m3"),
        # the FFN-up projection of the 14B model at 720p; the largest call
        _linear("video720p_ffn_int8", 75600, 5120, 13824),
        # loading a model: one of its FFN weights converted on the device
        _convert("convert_ffn_int8", 13824, 5120, "int8"),
    ]


# channel counts of the models the repository is measured on; drawn cases take these or any number between
WIDTHS = (1536, 4608, 5120, 8960, 13824, 15360)


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _width(rng, lo=256, hi=15360):
    if rng.random() < 0.5:
        return rng.choice([w for w in WIDTHS if lo <= w <= hi])
    return 8 * _log_int(rng, lo // 8, hi // 8)


def draw(rng):
    """One more case of the ranges that the listed ones stand for."""
    what = rng.choice(("rows", "text", "tokens", "video", "ragged", "tensor", "static", "ffn", "convert"))
    if what == "convert":
        return _convert(None, _log_int(rng, 256, 13824), _log_int(rng, 256, 5120), rng.choice(("int8", "e4m3")),
                        rng.choice(("bf16", "bf16", "fp16", "fp32")))
    if what == "ffn":
        k, n = 8 * _log_int(rng, 64, 640), 8 * _log_int(rng, 128, 1728)
        return _ffn(None, _log_int(rng, 256, min(37800, LARGEST // (2 * k * n))), k, n, rng.choice(("int8", "e4m3")))
    bias = rng.random() < 0.8
    if what == "ragged":  # any number of rows and channels, any module type
        m, k, n = _log_int(rng, 1, 16384), _log_int(rng, 40, 6000), _log_int(rng, 40, 6000)
        return _linear(None, m, k, n, "int8", "token", rng.choice(("bf16", "fp16", "fp32")), bias)
    k, n = _width(rng), _width(rng)
    m = _log_int(rng, *{"rows": (1, 127), "text": (128, 1024), "tokens": (1024, 12000), "video": (12000, 75600),
                        "tensor": (1, 12000), "static": (1, 12000)}[what])
    m = max(1, min(m, LARGEST // (k * n)))
    if what == "tensor":
        return _linear(None, m, k, n, rng.choice(("e5m2", "e4m3", "int8")), "tensor", "bf16", bias)
    if what == "static":
        return _linear(None, m, k, n, rng.choice(("e5m2", "e4m3")), "static", "bf16", bias)
    return _linear(None, m, k, n, rng.choice(("int8", "int8", "e4m3", "e5m2")), "token", "bf16", bias)


def _activations(g, m, k, dtype):
    x = torch.randn(m, k, generator=g, device=DEV)
    col = torch.ones(k, device=DEV)
    col[torch.randperm(k, generator=g, device=DEV)[: max(1, round(0.01 * k))]] = 20.0
    return x.mul_(col).to(dtype)


def _float_linear(g, k, n, dtype, bias=True):
    lin = nn.Linear(k, n, bias=bias, device="meta", dtype=dtype).to_empty(device=DEV)
    with torch.no_grad():
        lin.weight.copy_(torch.randn(n, k, generator=g, device=DEV).mul_(0.02))
        if bias:
            lin.bias.copy_(torch.randn(n, generator=g, device=DEV).mul_(0.01))
    return lin


def _dynamic_qconfig(fmt, scheme="token"):
    if scheme == "tensor":
        return get_default_dynamic_int8_qconfig() if fmt == "int8" else get_default_dynamic_fp8_qconfig(activation_dtype=ACT[fmt])
    if fmt == "int8":
        return get_dynamic_int8_per_token_act_per_channel_weight_qconfig()
    return get_dynamic_fp8_per_token_act_per_channel_weight_qconfig(activation_dtype=ACT[fmt])


@torch.no_grad()
def prepare(case, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    if case["kind"] == "convert":
        lin = _float_linear(g, case["k"], case["n"], DTYPES[case["dtype"]])
        lin.qconfig = _dynamic_qconfig(case["fmt"])
        return {"case": case, "linear": lin}
    if case["kind"] == "ffn":
        m, k, n = case["m"], case["k"], case["n"]
        model = nn.Sequential(_float_linear(g, k, n, torch.bfloat16), _float_linear(g, n, k, torch.bfloat16))
        quantize_dynamic(model, {"": _dynamic_qconfig(case["fmt"])})
        return {"case": case, "up": model[0], "down": model[1],
                "x": _activations(g, m, k, torch.bfloat16).view(1, m, k),
                "scale": torch.randn(1, 1, k, generator=g, device=DEV).mul_(0.2),
                "shift": torch.randn(1, 1, k, generator=g, device=DEV).mul_(0.2)}
    dtype = DTYPES[case["dtype"]]
    model = nn.Sequential(_float_linear(g, case["k"], case["n"], dtype, case["bias"]))
    x = _activations(g, case["m"], case["k"], dtype)
    if case["scheme"] == "static":
        prepare_static(model, {"": get_fp8_per_channel_weight_qconfig(activation_dtype=ACT[case["fmt"]])})
        model(x)  # calibration
        convert(model)
    else:
        quantize_dynamic(model, {"": _dynamic_qconfig(case["fmt"], case["scheme"])})
    return {"case": case, "linear": model[0], "x": x}


@torch.no_grad()
def run(state):
    kind = state["case"]["kind"]
    if kind == "linear":
        return state["linear"](state["x"])
    if kind == "ffn":
        up, down = state["up"], state["down"]
        qa = layernorm_quant(state["x"], 1 + state["scale"], state["shift"], LN_EPS, up)
        return down(gelu_tanh_quant(up(qa), down))
    q = Linear.from_float(state["linear"], reserve_float_weight=True)
    return {"qweight": q.qweight.view(torch.uint8), "weight_scale": q.weight_scale, "bias": q.bias}


def work(case):
    """Inputs read once, outputs written once, the multiply-adds of the matmuls."""
    k, n = case["k"], case["n"]
    if case["kind"] == "convert":
        return {"bytes": n * k * (BYTES[case["dtype"]] + 1) + 4 * n, "flops": 0}
    m = case["m"]
    if case["kind"] == "ffn":
        return {"bytes": 4 * m * k + 2 * n * k + 6 * (n + k) + 8 * k, "flops": 4 * m * n * k}
    e = BYTES[case["dtype"]]
    return {"bytes": e * m * (k + n) + n * k + (4 + (e if case["bias"] else 0)) * n, "flops": 2 * m * n * k}


def tolerance(case):
    # int8 sums are integers and every rounding behind them is specified; so are the statistics, scales and bytes of a weight
    if case["kind"] == "convert" or (case["kind"] == "linear" and case["fmt"] == "int8"):
        return "exact"
    # about four times the distance from the same operands multiplied in float64 with one rounding to bf16 at the end
    # (rel 3.6e-4 to 4.0e-4 and one bf16 step of 0.0078 at 2000 x 5120 x 5120, 4096 x 5120 x 5120 and 300 x 13824 x 1536)
    if case["kind"] == "linear":
        return {"rel": 1.6e-3, "max": 0.032}
    # ... from the same chain with LayerNorm, GELU (and FP8 sums) in float64: 2.4e-3 / 0.056 (e4m3), 3.1e-4 / 0.034 (int8)
    # at 1000 x 5120 x 13824; an activation that rounds to its neighbour moves its byte by one step of the format
    return {"rel": 1e-2, "max": 0.22} if case["fmt"] == "e4m3" else {"rel": 1.5e-3, "max": 0.14}
