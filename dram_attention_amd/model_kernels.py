"""The model's row-wise kernels (csrc/model_rows.hip) for tensors they take as they are;
llama.py keeps torch's operators for everything else (the CPU, autograd, odd layouts)."""

from __future__ import annotations

import torch

from . import _lib

_TYPES = (torch.bfloat16, torch.float16, torch.float32)


def takes(*tensors: torch.Tensor) -> bool:
    """Whether the kernels apply: contiguous, aligned GPU tensors of one type, and no
    autograd or autocast that would have to see the operation."""
    x = tensors[0]
    if not x.is_cuda or x.dtype not in _TYPES or torch.is_grad_enabled() or torch.is_autocast_enabled():
        return False
    return all(t.dtype == x.dtype and t.device == x.device and t.is_contiguous() and t.data_ptr() % 16 == 0
               for t in tensors)


def norm_fits(x: torch.Tensor) -> bool:
    row = x.shape[-1] * x.element_size()
    return row % 16 == 0 and row <= 32768


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float, add: torch.Tensor | None = None):
    """RMS norm of x, or of x + add; returns (norm, the sum or x)."""
    out = torch.empty_like(x)
    total = x if add is None else torch.empty_like(x)
    dim = x.shape[-1]
    _lib.check(
        _lib.load().da_rms_norm(
            x.data_ptr(), None if add is None else add.data_ptr(),
            None if add is None else total.data_ptr(), weight.data_ptr(), eps, out.data_ptr(),
            x.numel() // dim, dim, _lib.dtype_code(x.dtype), _lib.stream_ptr(x.device)),
        "da_rms_norm")
    return out, total


def rope_(xq: torch.Tensor, xk: torch.Tensor, table: torch.Tensor) -> None:
    """Rotate xq (1, S, Hq, D) and xk (1, S, Hkv, D) in place by the rows of table (S, D/2, 2)."""
    _lib.check(
        _lib.load().da_rope_rows(
            xq.data_ptr(), xq.stride(1), xk.data_ptr(), xk.stride(1), xq.shape[2], xk.shape[2], xq.shape[3],
            table.data_ptr(), xq.shape[1], _lib.dtype_code(xq.dtype), _lib.stream_ptr(xq.device)),
        "da_rope_rows")


def swiglu_(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up, in gate's place."""
    _lib.check(
        _lib.load().da_swiglu(gate.data_ptr(), up.data_ptr(), gate.data_ptr(), gate.numel(),
                              _lib.dtype_code(gate.dtype), _lib.stream_ptr(gate.device)),
        "da_swiglu")
    return gate
