"""Argument checks shared by the HIP binding wrappers.

They restate the reference's kernel-level TORCH_CHECKs (raised there as
RuntimeError) so that the bindings fail the same way:
``quantize_per_tensor_fp8.cu:164-167``, ``quantize_int8.cu:450-460``,
``dequantize_per_tensor_fp8.cu:88-97``, ``dequantize_int8.cu:191-202``.
"""
from __future__ import annotations

import os

import torch

from ... import _abi


def out_like(x: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    """An uninitialised contiguous tensor of x's shape and device (a plain
    torch.Tensor also where x is of a subclass). empty_like takes 1.0 us of
    host time, empty with a shape and a device 1.9."""
    if type(x) is torch.Tensor:
        return torch.empty_like(x, dtype=dtype, memory_format=torch.contiguous_format)
    return torch.empty(x.shape, dtype=dtype, device=x.device)


def check_cuda_contig(t: torch.Tensor, name: str) -> None:
    if not t.is_cuda:
        raise RuntimeError(f"{name} must be on CUDA")
    if not t.is_contiguous():
        raise RuntimeError(f"{name} must be contiguous")


def check_float_input(x: torch.Tensor, allow_f32: bool) -> int:
    check_cuda_contig(x, "x")
    if x.dtype == torch.float16 or x.dtype == torch.bfloat16 or (allow_f32 and x.dtype == torch.float32):
        return _abi.DTYPE_CODE[x.dtype]
    if allow_f32:
        raise RuntimeError("x must be torch.float16, torch.bfloat16, or torch.float32")
    raise RuntimeError("x must be torch.float16 or torch.bfloat16")


def check_scale(scale: torch.Tensor, q: torch.Tensor) -> torch.Tensor:
    if not scale.is_cuda:
        raise RuntimeError("scale must be on CUDA")
    if scale.dtype != torch.float32:
        raise RuntimeError("scale must be torch.float32")
    if scale.device != q.device:
        raise RuntimeError("scale must be on the same device as q")
    return scale.contiguous()


def check_out_dtype(dtype: torch.dtype) -> int:
    if dtype not in (torch.float16, torch.bfloat16):
        raise RuntimeError("out_dtype must be torch.float16 or torch.bfloat16")
    return _abi.DTYPE_CODE[dtype]


def watch_exchange(dev: torch.device) -> bool:
    """Whether CUBLADE_CHECK_EXCHANGE=1 is in the environment; if so, clears
    the status word of the stream's workspace where an earlier call left it set,
    so that check_exchange after the call tells of that call alone. The word is
    read first (which synchronises): a launch in front of every watched call
    would change how its workgroups start."""
    if os.environ.get("CUBLADE_CHECK_EXCHANGE", "") in ("", "0"):
        return False
    if _abi.tensor_quant_status(dev):
        _abi.clear_tensor_quant_status(dev)
    return True


def check_exchange(dev: torch.device, what: str) -> None:
    """Where watch_exchange returned True before a per-tensor quant:
    synchronise after it and raise RuntimeError if its workgroups' exchange
    timed out (the status word; cleared before raising). Off by default, so
    that calls stay asynchronous; a timed-out call's scale is NaN whenever a
    code is not exact, and later calls are exact either way."""
    if _abi.tensor_quant_status(dev):
        _abi.clear_tensor_quant_status(dev)
        raise RuntimeError(
            f"{what}: the workgroups of the one-launch per-tensor quant gave up waiting for "
            f"each other (exchange timed out; other work kept part of the grid off the GPU): "
            f"the result is not valid, repeat the call")
