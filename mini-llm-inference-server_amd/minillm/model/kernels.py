"""The decoder layer's kernels around its matrix products (csrc/norm.hip) and its products on few rows
(csrc/linear.hip), for the model's inference path.

`usable(x)` says whether a call may take them: a plain 16-bit CUDA tensor on the current device, gradients off, and
nothing active that follows torch's operations (tracing, compilation, autocast, function or dispatch modes, functorch
transforms, forward-mode derivatives).  Everything else keeps the torch expressions.  `bare(module, cls)` says whether
a submodule's `__call__` does nothing but its class's `forward`, so that a fused kernel may stand in for it.
"""

from __future__ import annotations

import math

import torch
from torch.autograd import forward_ad
from torch.nn.modules import module as _module

from .. import _native
from ..attention.hip_backend import FP8, HipBackend
from ..cache.paged import PagedKVCache, PagedStep

_DTYPES = (torch.bfloat16, torch.float16)
# what mllm_decoder_layer stands in for: a backend instance that overrides one of these is called instead
_BACKEND_CALLS = frozenset(("forward", "forward_rotary", "run_layer", "rope_append", "append", "attend"))
_transform = torch._C._functorch.peek_interpreter_stack  # the innermost active functorch transform, or None
_wrapped = torch._C._functorch.is_functorch_wrapped_tensor  # also of a wrapper that outlived its transform


def usable(x: torch.Tensor, dtype: torch.dtype | None = None) -> bool:
    """`dtype`: the type of the call's operands where x is not one of them.  Whether a compiler is at work is asked first:
    dynamo knows that answer while it traces and leaves out the rest, some of which it cannot trace.  Inside a transform
    (vmap and the like) any operand may be a wrapper without storage, not only x, so none is let through."""
    return (not torch.compiler.is_compiling() and type(x) is torch.Tensor and x.is_cuda
            and (dtype or x.dtype) in _DTYPES and not torch.is_grad_enabled() and not torch.is_autocast_enabled()
            and not torch._C._len_torch_dispatch_stack() and not torch._C._len_torch_function_stack()
            and _transform() is None and not _wrapped(x) and forward_ad._current_level < 0 and not torch.jit.is_tracing()
            and x.device.index == torch.cuda.current_device() and _native.available())


def bare(module: torch.nn.Module, cls: type) -> bool:
    d = module.__dict__
    return type(module) is cls and "forward" not in d \
        and not (d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"]
                 or _module._global_forward_hooks or _module._global_forward_pre_hooks
                 or _module._global_backward_hooks or _module._global_backward_pre_hooks)


def _rows_ok(t: torch.Tensor, like: torch.Tensor) -> bool:
    """A contiguous, 16-byte aligned operand of the same type and device, with storage."""
    return not _wrapped(t) and t.dtype == like.dtype and t.device == like.device and t.is_contiguous() \
        and t.data_ptr() % 16 == 0


def _plain_weight(w, like: torch.Tensor) -> bool:
    return type(w) in (torch.nn.Parameter, torch.Tensor) and _rows_ok(w, like)


MAX_GROUPS = (1 << 24) - 1  # workgroups of 256 threads one launch takes


def norm_ok(x: torch.Tensor, weight) -> bool:
    """Whether `rms_norm` takes x [..., D] (already `usable`) and its weight."""
    d = x.shape[-1]
    return d % 8 == 0 and 0 < x.numel() <= MAX_GROUPS * d and weight.shape == (d,) and _rows_ok(x, x) and _plain_weight(weight, x)


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


def rope_ok(positions: torch.Tensor, dtype: torch.dtype, half: int) -> bool:
    return (usable(positions, dtype) and positions.dtype == torch.int64 and positions.is_contiguous()
            and 0 < positions.numel() * half <= MAX_GROUPS * 256)


def rope_table(positions: torch.Tensor, inv_freq: torch.Tensor, dtype: torch.dtype):
    """cos, sin [..., 2 len(inv_freq)] of int64 positions."""
    half = inv_freq.shape[0]
    cos = torch.empty((*positions.shape, 2 * half), dtype=dtype, device=positions.device)
    sin = torch.empty_like(cos)
    _native.lib().call("mllm_rope_table", positions.data_ptr(), positions.numel(), inv_freq.data_ptr(), half,
                       _native.dtype_code(dtype), cos.data_ptr(), sin.data_ptr(), _native.stream_ptr(positions.device))
    return cos, sin


def sum_ok(x: torch.Tensor, y: torch.Tensor) -> bool:
    return type(y) is torch.Tensor and y.shape == x.shape and _rows_ok(y, x)


def silu_mul_ok(gate: torch.Tensor, up: torch.Tensor) -> bool:
    return usable(gate) and sum_ok(gate, up) and _rows_ok(gate, gate) and gate.numel() % 8 == 0 \
        and gate.numel() <= MAX_GROUPS * 2048


def silu_mul(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up with one rounding."""
    out = torch.empty_like(gate)
    _native.lib().call("mllm_silu_mul", gate.data_ptr(), up.data_ptr(), gate.numel(), _native.dtype_code(gate.dtype),
                       out.data_ptr(), _native.stream_ptr(gate.device))
    return out


# ---------------------------------------------------------------- linear layers of few rows

SMALL_ROWS = 64  # rows of x the kernels take
CHUNK = 256  # K granularity


def small_rows(x: torch.Tensor) -> bool:
    """Whether x [..., K] has few enough rows for these kernels.  The line lies at 64, what their accumulators and LDS are
    laid out for; up to it each measured faster than the library product (csrc/linear.hip), with q, k, v and gate,
    up sharing launches on top."""
    return type(x) is torch.Tensor and 0 < x.numel() <= SMALL_ROWS * x.shape[-1] and _rows_ok(x, x)


def weights_ok(like: torch.Tensor, k: int, *linears) -> bool:
    """Whether the few-row kernels take these layers for operands of `k` columns with the type and device of `like`."""
    if k % CHUNK or k >= 1 << 24:
        return False
    for m in linears:
        # taken from the registered parameters; a layer that holds them as plain attributes (a data-parallel replica)
        # is called
        params = m.__dict__["_parameters"]
        if not bare(m, torch.nn.Linear) or params.get("bias", m) is not None or params.get("weight") is None:
            return False
        w = params["weight"]
        if w.shape[1] != k or w.shape[0] % 16 or w.shape[0] >= 1 << 28 or not _plain_weight(w, like):
            return False
    return True


def _partial(x: torch.Tensor, weights) -> tuple[torch.Tensor, int, int]:
    k = x.shape[-1]
    m = x.numel() // k
    rows = [w.shape[0] for w in weights]
    ks = _native.lib().fn("mllm_linear_ksplit")(k, *rows, *(0,) * (4 - len(rows)))
    part = torch.empty(ks * m * sum(rows), dtype=torch.float32, device=x.device)
    args = []
    for w in weights:
        args += (w.data_ptr(), w.shape[0])
    args += (None, 0) * (3 - len(weights))
    _native.lib().call("mllm_linear_partial", x.data_ptr(), m, k, *args, ks, part.data_ptr(),
                       _native.dtype_code(x.dtype), _native.stream_ptr(x.device))
    return part, ks, m


def linear(x: torch.Tensor, *weights, residual: torch.Tensor | None = None) -> torch.Tensor:
    """x . w^T of each weight side by side, [..., sum of rows] (plus `residual`, of that shape)."""
    part, ks, m = _partial(x, weights)
    n = part.numel() // (ks * m)
    out = torch.empty((*x.shape[:-1], n), dtype=x.dtype, device=x.device)
    _native.lib().call("mllm_sum_partials", part.data_ptr(), ks, m, n,
                       None if residual is None else residual.data_ptr(), _native.dtype_code(x.dtype), out.data_ptr(),
                       _native.stream_ptr(x.device))
    return out


def linear_add_norm(x: torch.Tensor, weight: torch.Tensor, residual: torch.Tensor, norm: torch.Tensor, eps: float):
    """(residual + x . w^T, its RMSNorm)."""
    part, ks, m = _partial(x, (weight,))
    total, out = torch.empty_like(residual), torch.empty_like(residual)
    _native.lib().call("mllm_sum_partials_norm", part.data_ptr(), ks, residual.data_ptr(), norm.data_ptr(), m,
                       weight.shape[0], eps, _native.dtype_code(x.dtype), total.data_ptr(), out.data_ptr(),
                       _native.stream_ptr(x.device))
    return total, out


def linear_swiglu(x: torch.Tensor, gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """silu(x . gate^T) * (x . up^T)."""
    k, n = x.shape[-1], gate.shape[0]
    out = torch.empty((*x.shape[:-1], n), dtype=x.dtype, device=x.device)
    _native.lib().call("mllm_linear_swiglu", x.data_ptr(), x.numel() // k, k, gate.data_ptr(), up.data_ptr(), n,
                       _native.dtype_code(x.dtype), out.data_ptr(), _native.stream_ptr(x.device))
    return out


def decoder_layer(layer, x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, kv_cache) -> torch.Tensor | None:
    """A decoder layer of a paged step of few rows in one host call (mllm_decoder_layer), or None when it does not apply:
    another cache or backend, hooks, or operands its checks would refuse.  `layer` has passed `_small_ok`; the launches
    are those of the submodules one after the other."""
    if type(kv_cache) is not PagedStep or type(kv_cache.cache) is not PagedKVCache or x.dim() != 3 or x.shape[0] != 1:
        return None
    attn, norm1, norm2 = layer.self_attn, layer.input_layernorm, layer.post_attention_layernorm
    backend, cfg, cache, meta = attn.backend, attn.config, kv_cache.cache, kv_cache.meta
    if type(backend) is not HipBackend or not backend.fuse_rotary or backend.overlap_mixed \
            or not _BACKEND_CALLS.isdisjoint(backend.__dict__):
        return None
    n, d = x.shape[1], x.shape[2]
    h, hkv, dh = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    wq, wk, wv = attn.q_proj, attn.k_proj, attn.v_proj
    if not (bare(norm1, type(norm2)) and norm_ok(x, norm1.weight) and weights_ok(x, d, wq, wk, wv)
            and weights_ok(x, h * dh, attn.o_proj)):
        return None
    wq, wk, wv = wq.weight, wk.weight, wv.weight
    if wq.shape[0] != h * dh or wk.shape[0] != hkv * dh or wv.shape[0] != hkv * dh:
        return None
    if cos.shape != (1, n, dh) or sin.shape != cos.shape or not (_rows_ok(cos, x) and _rows_ok(sin, x)):
        return None
    i = attn.layer_idx
    kc, vc = cache.k[i], cache.v[i]
    if not (kc.dim() == 4 and kc.shape == vc.shape and kc.dtype == vc.dtype and kc.device == vc.device == x.device
            and kc.shape[2] == hkv and kc.shape[3] == dh and kc.shape[1] == meta.block_size and kc.is_contiguous()
            and vc.is_contiguous() and n == meta.query_start_loc[-1]):
        return None
    ks, vs = (cache.k_scale[i], cache.v_scale[i]) if cache.quantized else (1.0, 1.0)
    if kc.dtype == FP8:
        if not (0 < ks < math.inf and 0 < vs < math.inf):
            return None
    elif kc.dtype != x.dtype or ks != 1.0 or vs != 1.0:
        return None
    lib, mlp = _native.lib(), layer.mlp
    gate = mlp.gate_proj.weight
    ffn = gate.shape[0]
    scratch = torch.empty(lib.fn("mllm_decoder_layer_scratch_bytes")(n, d, ffn, h, hkv, dh), dtype=torch.uint8,
                          device=x.device)
    step = backend.layer_step(meta, n, h, x.dtype, kc)
    out = torch.empty_like(x)
    lib.call("mllm_decoder_layer", step, x.data_ptr(), d, norm1.weight.data_ptr(), norm1.eps, wq.data_ptr(), wk.data_ptr(),
             wv.data_ptr(), attn.o_proj.weight.data_ptr(), norm2.weight.data_ptr(), norm2.eps, gate.data_ptr(),
             mlp.up_proj.weight.data_ptr(), mlp.down_proj.weight.data_ptr(), ffn, cos.data_ptr(), sin.data_ptr(),
             dh, kc.data_ptr(), vc.data_ptr(), ks, vs, scratch.data_ptr(), scratch.numel(), out.data_ptr(),
             _native.stream_ptr(x.device))
    return out
