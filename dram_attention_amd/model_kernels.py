"""The model's row-wise kernels (csrc/model_rows.hip) and its linear layers for one token
(csrc/decode_linear.hip), for tensors they take as they are; llama.py keeps torch's
operators for everything else (the CPU, autograd, odd layouts)."""

from __future__ import annotations

import torch
from torch import nn
from torch.autograd import forward_ad
from torch.nn.modules import module as nn_module
from torch.utils._device import DeviceContext

from . import _lib

# (asked several times for every layer of a token)
_transform_level = torch._C._functorch.maybe_current_level
_dispatch_modes, _function_modes = torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack
_tracing_state = torch._C._get_tracing_state


def unobserved() -> bool:
    """Whether nothing but the tensors' values depends on which operators run: no forward-mode
    differentiation (which torch.no_grad leaves on), vmap or other transform, dispatch or
    function mode, tracer or compiler would have to see them."""
    # (the compiler first: it cannot follow the other questions)
    return (not torch.compiler.is_compiling()
            and forward_ad._current_level < 0 and _transform_level() is None
            and not _dispatch_modes() and _tracing_state() is None
            and not (_function_modes() and _function_mode_watches()))


def _function_mode_watches() -> bool:
    """Whether a function mode other than torch.device(...) and torch.set_default_device, which
    only say where new tensors are born, is on."""
    return any(type(torch._C._get_function_stack_at(i)) is not DeviceContext for i in range(_function_modes()))


def takes(*tensors: torch.Tensor) -> bool:
    """Whether the kernels apply: plain, contiguous, aligned GPU tensors of one type, and no
    autograd, autocast or transform that would have to see the operation."""
    return (tensors[0].is_cuda and not torch.is_grad_enabled() and not torch.is_autocast_enabled() and unobserved()
            and _lib.host().alike(*tensors))


def norm_fits(x: torch.Tensor, weight: torch.Tensor) -> bool:
    row = x.shape[-1] * x.element_size()
    return weight.shape == x.shape[-1:] and x.numel() > 0 and row % 16 == 0 and row <= 32768


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


def bare(*modules: nn.Module) -> bool:
    """Whether calling these modules does nothing but their class's forward: nobody hooked
    them or gave one of them a forward of its own."""
    if nn_module._global_forward_hooks or nn_module._global_forward_pre_hooks:
        return False
    for m in modules:
        if m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__:
            return False
    return True


def plain_linears(*modules: nn.Module) -> bool:
    """Whether the outputs of these modules are fresh tensors that nobody else holds, so
    that they may be changed in place: torch's own nn.Linear, unwatched."""
    return all(type(m) is nn.Linear for m in modules) and bare(*modules)


MAX_LINEAR_ROW = 60 * 1024  # bytes of an input row the one-token layers hold in LDS


def linears_fit(x: torch.Tensor, *linears) -> tuple | None:
    """The weights of these nn.Linear modules, if the one-token layers may stand for them (x: any
    tensor of the step, for its type and device), else None.  Each as a module or as (module,
    outputs, inputs), where only these sizes will do."""
    # (hooks first: pruning and weight normalisation keep the class, move the parameter and put
    # the weight together in a pre-hook)
    if nn_module._global_forward_hooks or nn_module._global_forward_pre_hooks:
        return None
    args = []
    for m in linears:
        args += m if type(m) is tuple else (m, -1, -1)
    return _lib.host().linears(x, nn.Linear, MAX_LINEAR_ROW, *args)


def row_fits(row, x: torch.Tensor, n: int) -> bool:
    """Whether ``row``, which any module may have made, is what the one-token layers read: n
    elements of x's type on x's device, in place one after the other."""
    return (type(row) is torch.Tensor and row.dtype is x.dtype and row.device == x.device and row.numel() == n
            and row.is_contiguous() and row.data_ptr() % 16 == 0)


def linear_qkv_rope(x, norm, wq, wk, wv, n_heads, n_kv_heads, head_dim, rope_row):
    """Rotated queries and keys, and values, of one token: (1,1,Hq,D), (1,1,Hkv,D) x 2."""
    return _lib.host().qkv_rope(x, norm.weight, norm.eps, wq, wk, wv, n_heads, n_kv_heads, head_dim, rope_row,
                                _lib.stream_ptr(x.device))


def linear_swiglu(x, norm, w1, w3):
    """silu(w1 n) * (w3 n), n the norm of x (1, 1, dim)."""
    out = torch.empty(1, 1, w1.shape[0], dtype=x.dtype, device=x.device)
    _lib.check(
        _lib.load().da_linear_swiglu(
            x.data_ptr(), norm.weight.data_ptr(), norm.eps, x.shape[-1], w1.data_ptr(), w3.data_ptr(),
            w1.shape[0], out.data_ptr(), _lib.dtype_code(x.dtype), _lib.stream_ptr(x.device)),
        "da_linear_swiglu")
    return out


def linear_add(x, w, residual):
    """residual + w x for one token; x of any shape with w.shape[1] elements."""
    out = torch.empty_like(residual)
    _lib.check(
        _lib.load().da_linear_add(
            x.data_ptr(), w.shape[1], w.data_ptr(), w.shape[0], residual.data_ptr(), out.data_ptr(),
            _lib.dtype_code(x.dtype), _lib.stream_ptr(x.device)),
        "da_linear_add")
    return out


def block_tail(attended, wo, x, norm, w1, w3, w2):
    """The rest of a block behind attention's output, residuals included, as one call."""
    return _lib.host().block_tail(attended, wo, x, norm.weight, norm.eps, w1, w3, w2, _lib.stream_ptr(x.device))


def linear_logits(x, norm, w):
    """fp32 logits (1, 1, vocab) of the normed row x (1, 1, dim)."""
    out = torch.empty(1, 1, w.shape[0], dtype=torch.float32, device=x.device)
    _lib.check(
        _lib.load().da_linear_logits(
            x.data_ptr(), norm.weight.data_ptr(), norm.eps, x.shape[-1], w.data_ptr(), w.shape[0],
            out.data_ptr(), _lib.dtype_code(x.dtype), _lib.stream_ptr(x.device)),
        "da_linear_logits")
    return out


def is_token(token, logits: torch.Tensor) -> bool:
    """Whether the arg-max kernel may write ``token``: one plain int64 on the logits' device."""
    return (type(token) is torch.Tensor and token.dtype == torch.int64 and token.numel() == 1
            and token.device == logits.device)


def argmax_into(logits: torch.Tensor, token: torch.Tensor) -> None:
    """token (one int64) = index of the largest of the contiguous fp32 logits."""
    _lib.check(
        _lib.load().da_argmax(logits.data_ptr(), logits.numel(), token.data_ptr(),
                              _lib.stream_ptr(logits.device)),
        "da_argmax")
