"""The decoder layer's kernels around its matrix products (csrc/norm.hip), for the model's inference path.

`usable(x)` says whether a call may take them: a plain 16-bit CUDA tensor on the current device, gradients off, and
nothing active that follows torch's operations (tracing, compilation, autocast, function or dispatch modes, functorch
transforms, forward-mode derivatives).  Everything else keeps the torch expressions.  `bare(module, cls)` says whether
a submodule's `__call__` does nothing but its class's `forward`, so that a fused kernel may stand in for it.
"""

from __future__ import annotations

import torch
from torch.autograd import forward_ad
from torch.nn.modules import module as _module

from .. import _native

_DTYPES = (torch.bfloat16, torch.float16)
_wrapped = torch._C._functorch.is_functorch_wrapped_tensor
_HOOKS = ("_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks")


def usable(x: torch.Tensor) -> bool:
    return (type(x) is torch.Tensor and x.is_cuda and x.dtype in _DTYPES and not torch.is_grad_enabled()
            and not torch.is_autocast_enabled() and not torch._C._len_torch_dispatch_stack()
            and not torch._C._len_torch_function_stack() and not _wrapped(x) and forward_ad._current_level < 0
            and not torch.compiler.is_compiling() and not torch.jit.is_tracing()
            and x.device.index == torch.cuda.current_device() and _native.LIB_PATH.exists())


def bare(module: torch.nn.Module, cls: type) -> bool:
    if type(module) is not cls or "forward" in module.__dict__:
        return False
    if any(getattr(module, h) for h in _HOOKS):
        return False
    return not (_module._global_forward_hooks or _module._global_forward_pre_hooks or _module._global_backward_hooks
                or _module._global_backward_pre_hooks)


def _rows_ok(t: torch.Tensor, like: torch.Tensor) -> bool:
    """A contiguous, 16-byte aligned operand of the same type and device."""
    return t.dtype == like.dtype and t.device == like.device and t.is_contiguous() and t.data_ptr() % 16 == 0


def _plain_weight(w, like: torch.Tensor) -> bool:
    return type(w) in (torch.nn.Parameter, torch.Tensor) and _rows_ok(w, like)


def norm_ok(x: torch.Tensor, weight) -> bool:
    """Whether `rms_norm` takes x [..., D] (already `usable`) and its weight."""
    d = x.shape[-1]
    return d % 8 == 0 and x.numel() > 0 and weight.shape == (d,) and _rows_ok(x, x) and _plain_weight(weight, x)


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    out = torch.empty_like(x)
    d = x.shape[-1]
    _native.lib().call("mllm_rms_norm", x.data_ptr(), None, weight.data_ptr(), x.numel() // d, d, eps,
                       _native.dtype_code(x.dtype), None, out.data_ptr(), _native.stream_ptr(x.device))
    return out


def add_rms_norm(x: torch.Tensor, y: torch.Tensor, weight: torch.Tensor, eps: float):
    """(x + y, its norm) in one launch."""
    total, out = torch.empty_like(x), torch.empty_like(x)
    d = x.shape[-1]
    _native.lib().call("mllm_rms_norm", x.data_ptr(), y.data_ptr(), weight.data_ptr(), x.numel() // d, d, eps,
                       _native.dtype_code(x.dtype), total.data_ptr(), out.data_ptr(), _native.stream_ptr(x.device))
    return total, out


def sum_ok(x: torch.Tensor, y: torch.Tensor) -> bool:
    return type(y) is torch.Tensor and y.shape == x.shape and _rows_ok(y, x)


def silu_mul_ok(gate: torch.Tensor, up: torch.Tensor) -> bool:
    return usable(gate) and sum_ok(gate, up) and _rows_ok(gate, gate) and gate.numel() % 8 == 0


def silu_mul(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up with one rounding."""
    out = torch.empty_like(gate)
    _native.lib().call("mllm_silu_mul", gate.data_ptr(), up.data_ptr(), gate.numel(), _native.dtype_code(gate.dtype),
                       out.data_ptr(), _native.stream_ptr(gate.device))
    return out
