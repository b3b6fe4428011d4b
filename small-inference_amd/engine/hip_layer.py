"""The decoder layer's operations around the paged attention on MI355X through libsmallinf_hip.so: RMSNorm, the
projections of a few tokens fused with the operations next to them, rotary embedding and SwiGLU (reference
engine/model.py:101-175, there about 30 torch operations a layer).

Each function takes bf16 GPU tensors with a contiguous last dimension, unchecked beyond what the library checks:
`supported` (a whole layer) or `rows_ok` (a norm) comes first, and the model runs its torch operations where they say no.
"""

from __future__ import annotations

import ctypes
import functools

import torch
import torch.nn.functional as F
from torch.utils._device import DeviceContext

from . import _hip

RESIDUAL, ROPE, SILU = 0, 1, 2  # SIPA_LINEAR_*

# Up to here a layer's projections run the fused kernels; larger batches go to the GEMM library with the fused
# operations around it. A 0.5B layer's projections and what they fuse (us, fused against library): 64 tokens 29 / 54,
# 256 41 / 59, 544 57 / 64, 1024 81 / 84.
MAX_TOKENS = 1024
# The gated projection goes to the library above this many operations, where its large tiles are better. A whole layer (us,
# fused against library): 0.5B at 768 tokens (13.4 GFLOP) 81 / 87, 832 (14.5) 88 / 92, 896 (15.6) 94 / 87, 960 96 / 97, 1024
# (17.9) 97 / 96; 1.5B at 224 (12.3) 90 / 88, 256 (14.1) 95 / 93, 288 (15.9) 97 / 92, 320 101 / 97, 448 (24.7) 141 / 121.
MAX_GATED_FLOPS = 15e9


_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _ok(device: int, *wanted: tuple[torch.Tensor, tuple[int, ...]]) -> bool:
    """Whether every (tensor, shape) is a contiguous bf16 tensor of that shape on the device, 16-byte aligned."""
    for t, shape in wanted:
        if type(t) not in _PLAIN or t.dtype is not torch.bfloat16 or t.get_device() != device or t.shape != shape or \
                not t.is_contiguous() or t.data_ptr() % 16:
            return False
    return True


# looked up once: a layer asks them all for every call
_inference, _autocast, _compiling = torch.is_inference_mode_enabled, torch.is_autocast_enabled, torch.compiler.is_compiling
_tracing, _transform = torch._C._is_tracing, torch._C._functorch.peek_interpreter_stack
_dispatch_modes, _function_modes = torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack


def _plain() -> bool:
    """Whether torch operations would just run: under torch.inference_mode (the kernels record nothing for autograd, and
    saved-tensor hooks do not reach them there), not under autocast, whose type the products' results have, and with
    nobody between who is to see each operation: vmap, grad or jvp, tracing or compilation, a dispatch mode, or a function
    mode other than the default device's."""
    if not _inference() or _autocast() or _compiling() or _tracing() or _transform() is not None or \
            _dispatch_modes():
        return False
    n = _function_modes()
    return n == 0 or all(type(torch._C._get_function_stack_at(i)) is DeviceContext for i in range(n))


def rows_ok(x: torch.Tensor, norm_weight: torch.Tensor) -> bool:
    """Whether rms_norm can run on rows x [T, K], and stand for the torch operations."""
    if not (x.is_cuda and x.dim() == 2 and _plain()):
        return False
    T, K = x.shape
    return K % 8 == 0 and K <= 8192 and _ok(x.get_device(), (x, (T, K)), (norm_weight, (K,)))


def supported(x: torch.Tensor, w, rot, heads: int, head_dim: int) -> bool:
    """Whether the layer w (engine.model.Layer) with `heads` query, key and value heads can run on hidden states
    x [T, hidden] with the kernels below: bf16, contiguous, 16-byte aligned tensors of one GPU whose sizes are whole
    tiles. The model's torch operations serve everything else, and raise their own errors for sizes that disagree."""
    if not rows_ok(x, w.input_norm):
        return False
    T, hidden = x.shape
    dev, width, inter, attn = x.get_device(), heads * head_dim, w.down_w.shape[-1], w.o_w.shape[-1]
    cos, sin = rot
    if max(width, inter, attn) > 1 << 20 or T * max(width, inter) >= 1 << 34:  # the library's limits
        return False
    return (head_dim % 16 == 0 and hidden % 64 == 0 and inter % 64 == 0 and attn % 64 == 0 and
            _ok(dev, (w.qkv_w, (width, hidden)), (w.qkv_b, (width,)), (w.o_w, (hidden, attn)), (w.post_norm, (hidden,)),
                (w.gate_up_w, (2 * inter, hidden)), (w.down_w, (hidden, inter)), (cos, (T, 1, head_dim)),
                (sin, (T, 1, head_dim))))


def attention_ok(attn: torch.Tensor, x: torch.Tensor, w) -> bool:
    """Whether layer_out can read attn, what a cache's attend returned for a supported layer w: bf16 rows [T, o_w's
    features] on x's device, 16-byte aligned. The kernels take its size for the projection's, so one that differs would
    be read past its end."""
    return type(attn) in _PLAIN and attn.dtype is torch.bfloat16 and attn.get_device() == x.get_device() and \
        attn.shape == (x.shape[0], w.o_w.shape[1]) and attn.stride(1) == 1 and attn.stride(0) >= attn.shape[1] and \
        attn.stride(0) % 8 == 0 and attn.data_ptr() % 16 == 0


@functools.lru_cache(maxsize=1024)
def _linear_scratch(epilogue: int, norm: bool, T: int, K: int, N: int, head_dim: int, num_splits: int, tile: int) -> int:
    p = _hip.LinearParams(struct_size=ctypes.sizeof(_hip.LinearParams), epilogue=epilogue, num_tokens=T, in_features=K,
                          out_features=N, head_dim=head_dim, norm_weight=16 if norm else None, num_splits=num_splits,
                          tile=tile)
    n = _hip.lib().sipa_linear_scratch_bytes(ctypes.byref(p))
    if n < 0:
        _hip.check(n, "fused_linear")
    return n


def fused_linear(x: torch.Tensor, weight: torch.Tensor, epilogue: int, *, norm_weight: torch.Tensor | None = None,
                 eps: float = 0.0, bias: torch.Tensor | None = None, residual: torch.Tensor | None = None,
                 rot: tuple[torch.Tensor, torch.Tensor] | None = None, head_dim: int = 0, rot_channels: int = 0,
                 num_splits: int = 0, tile: int = 0, store: tuple | None = None,
                 counters: torch.Tensor | None = None, clear: torch.Tensor | None = None) -> torch.Tensor:
    """epilogue(norm(x) W^T) in one launch (sipa_fused_linear): x [T, K], weight [N, K]; RESIDUAL adds bias and
    residual, ROPE adds bias and rotates the first rot_channels channels by rot = (cos, signed sin), SILU multiplies
    the second half of the channels by silu of the first. num_splits, tile: 0 for the library's choice. store (ROPE):
    PagedKVCache.store_target's tuple; the K and V channels then go to the pools and are undefined in the result. A K that
    several workgroups share needs merge counters at zero: `counters`, int32, which an earlier launch was given as `clear`,
    or new ones from a launch of their own (None)."""
    T, K = x.shape
    N = weight.shape[0]
    out = torch.empty(T, N // 2 if epilogue == SILU else N, device=x.device, dtype=torch.bfloat16)
    stream = _hip.stream_of(x)
    n = _linear_scratch(epilogue, norm_weight is not None, T, K, N, head_dim, num_splits, tile)
    scratch = None
    if n:
        scratch = torch.empty(n, device=x.device, dtype=torch.uint8)
        if counters is None:  # one a tile, and a tile has 32 x 32 fp32 sums or more
            counters = torch.zeros(n // 4096, device=x.device, dtype=torch.int32)
    p = _hip.LinearParams(ctypes.sizeof(_hip.LinearParams), epilogue, T, K, N, head_dim, rot_channels, eps,
                          x.data_ptr(), x.stride(0), weight.data_ptr(), _hip.ptr(norm_weight), _hip.ptr(bias),
                          _hip.ptr(residual), residual.stride(0) if residual is not None else 0, out.data_ptr(),
                          out.stride(0), *((rot[0].data_ptr(), rot[1].data_ptr()) if rot is not None else (None, None)),
                          num_splits, tile, _hip.ptr(scratch), n, _hip.ptr(counters), *(store or ()))
    if clear is not None:
        p.clear, p.clear_count = clear.data_ptr(), clear.numel()
    _hip.check(_hip.lib().sipa_fused_linear(ctypes.byref(p), stream), "fused_linear")
    return out


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float, add: torch.Tensor | None = None):
    """RMSNorm of x's rows, or of s = x + add; returns the normalised rows, with s when add is given. One launch."""
    T, K = x.shape
    out = torch.empty(T, K, device=x.device, dtype=torch.bfloat16)
    s = torch.empty_like(out) if add is not None else None
    _hip.check(_hip.lib().sipa_rms_norm(x.data_ptr(), x.stride(0), _hip.ptr(add), add.stride(0) if add is not None
                                        else 0, weight.data_ptr(), eps, _hip.ptr(s), K, out.data_ptr(), K, T, K,
                                        _hip.stream_of(x)), "rms_norm")
    return out if add is None else (out, s)


def rope_(x: torch.Tensor, rot: tuple[torch.Tensor, torch.Tensor], heads: int, head_dim: int) -> None:
    """Rotary embedding in place on the first `heads` heads of rows x [T, >= heads * head_dim]. One launch."""
    _hip.check(_hip.lib().sipa_rope(x.data_ptr(), x.stride(0), rot[0].data_ptr(), rot[1].data_ptr(), x.shape[0],
                                    heads, head_dim, _hip.stream_of(x)), "rope")


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    """silu(first half) * second half of the channels. One launch."""
    T, I = gate_up.shape[0], gate_up.shape[1] // 2
    out = torch.empty(T, I, device=gate_up.device, dtype=torch.bfloat16)
    _hip.check(_hip.lib().sipa_silu_mul(gate_up.data_ptr(), gate_up.stride(0), out.data_ptr(), I, T, I,
                                        _hip.stream_of(gate_up)), "silu_mul")
    return out


def layer_qkv(x: torch.Tensor, w, eps: float, rot, rotated: int, head_dim: int, store: tuple | None = None) -> torch.Tensor:
    """[T, heads * head_dim]: the fused projection of the normalised x, its first `rotated` heads (queries and keys)
    rotated; with store, K and V in the cache's pools instead. One launch, up to MAX_TOKENS."""
    return fused_linear(x, w.qkv_w, ROPE, norm_weight=w.input_norm, eps=eps, bias=w.qkv_b, rot=rot, head_dim=head_dim,
                        rot_channels=rotated * head_dim, store=store)


def layer_qkv_large(x: torch.Tensor, w, eps: float, rot, rotated: int, head_dim: int) -> torch.Tensor:
    """The same for more tokens, the product in the GEMM library: three launches."""
    qkv = F.linear(rms_norm(x, w.input_norm, eps), w.qkv_w, w.qkv_b)
    rope_(qkv, rot, rotated, head_dim)
    return qkv


@functools.lru_cache(maxsize=1024)
def _layer_out_scratch(T: int, hidden: int, attn_features: int, inter: int) -> int:
    p = _hip.LayerOutParams(ctypes.sizeof(_hip.LayerOutParams), T, hidden, attn_features, inter)
    n = _hip.lib().sipa_layer_out_scratch_bytes(ctypes.byref(p))
    if n < 0:
        _hip.check(n, "layer_out")
    return n


def layer_out(x: torch.Tensor, attn: torch.Tensor, w, eps: float) -> torch.Tensor:
    """x + attn W_o, then that plus its MLP: three launches from one call, up to MAX_TOKENS and MAX_GATED_FLOPS."""
    T, hidden = x.shape
    inter = w.down_w.shape[1]
    if T > MAX_TOKENS:
        n, h = rms_norm(x, w.post_norm, eps, add=F.linear(attn, w.o_w))
        return h + F.linear(silu_mul(F.linear(n, w.gate_up_w)), w.down_w)
    if 4.0 * T * hidden * inter > MAX_GATED_FLOPS:
        counters = torch.empty(_hip.LAYER_COUNTERS, device=x.device, dtype=torch.int32)
        h = fused_linear(attn, w.o_w, RESIDUAL, residual=x, clear=counters)
        act = silu_mul(F.linear(rms_norm(h, w.post_norm, eps), w.gate_up_w))
        return fused_linear(act, w.down_w, RESIDUAL, residual=h, counters=counters)
    out = torch.empty(T, hidden, device=x.device, dtype=torch.bfloat16)
    nbytes = _layer_out_scratch(T, hidden, attn.shape[1], inter)
    # the sums and then the merge counters of split projections, in memory of this call's own: what a graph holds of them
    # is its own too
    scratch = torch.empty(nbytes + 4 * _hip.LAYER_COUNTERS, device=x.device, dtype=torch.uint8)
    p = _hip.LayerOutParams(ctypes.sizeof(_hip.LayerOutParams), T, hidden, attn.shape[1], inter, eps, x.data_ptr(),
                            x.stride(0), attn.data_ptr(), attn.stride(0), w.o_w.data_ptr(), w.post_norm.data_ptr(),
                            w.gate_up_w.data_ptr(), w.down_w.data_ptr(), out.data_ptr(), scratch.data_ptr(), nbytes,
                            scratch.data_ptr() + nbytes)
    _hip.check(_hip.lib().sipa_layer_out(ctypes.byref(p), _hip.stream_of(x)), "layer_out")
    return out
