"""Leaf quantisers: a tensor and the scale of each of its rows in, quantised values out.

Same names and argument meaning as dax/quant/nn/quantized/functional.py:4-20; the work is
done by the HIP kernels ``daxq_quantize_rows_*`` (int8: reciprocal-multiply, round half to
even, clamp; e4m3fn / e5m2: true division, clamp to +-448 / +-57344, round to nearest even).
A scale of one element (per-tensor scheme) is read as it is (``daxq_quantize_tensor``).
"""
import torch
from torch import Tensor

from .... import ops

FP8_ALLOWED_DTYPES = (
    torch.float8_e4m3fn,
    torch.float8_e5m2,
)


def _quantize(x: Tensor, scale: Tensor, fmt: str) -> Tensor:
    if scale.numel() == 1 and 0 < x.shape[-1] <= ops.MAX_TENSOR_QUANT_K:
        return ops.quantize_tensor(x.reshape(-1, x.shape[-1]), scale.reshape(1).to(torch.float32), fmt, False)[0]
    x2, s = _rows_and_scale(x, scale)
    return getattr(ops, "quantize_rows_" + fmt)(x2, s)


def _rows_and_scale(x: Tensor, scale: Tensor):
    """Flattens x to [rows, K] and gives every row its scale (scale broadcasts against x
    with a trailing dimension of 1, or is a single value)."""
    k = x.shape[-1]
    x2 = x.reshape(-1, k)
    if scale.numel() == 1:
        return x2, ops.broadcast_f32(scale.reshape(1).to(torch.float32).contiguous(), x2.shape[0])
    else:
        if scale.shape[-1] != 1 and scale.dim() == x.dim():
            raise NotImplementedError("daxq leaf quantisers take one scale per row (or one per tensor)")
        s = scale.to(torch.float32).expand(*x.shape[:-1], 1).reshape(-1)
    return x2, s.contiguous()


def quantize_to_fp8(x: Tensor, scale: Tensor, dtype: torch.dtype) -> Tensor:
    if dtype not in FP8_ALLOWED_DTYPES:
        raise NotImplementedError(f"daxq implements float8_e4m3fn and float8_e5m2, got {dtype}")
    return _quantize(x, scale, "e4m3" if dtype == torch.float8_e4m3fn else "e5m2").view(dtype).view(x.shape)


def quantize_to_int8(x: Tensor, scale: Tensor, dtype: torch.dtype) -> Tensor:
    if dtype != torch.int8:
        raise NotImplementedError(f"daxq implements int8 only, got {dtype}")
    return _quantize(x, scale, "i8").view(x.shape)
