"""The decoder layer's operations around the paged attention on MI355X through libsmallinf_hip.so: RMSNorm, the
projections of a few tokens fused with the operations next to them, rotary embedding and SwiGLU (reference
engine/model.py:101-175, there about 30 torch operations a layer).

Each function takes bf16 GPU tensors with a contiguous last dimension, unchecked beyond what the library checks:
`supported` (a whole layer) or `rows_ok` (a norm) comes first, and the model runs its torch operations where they say no.
"""

from __future__ import annotations

import ctypes

import torch
import torch.nn.functional as F

from . import _hip
from .hip_decode import reserve_workspace

RESIDUAL, ROPE, SILU = 0, 1, 2  # SIPA_LINEAR_*
# Up to here the projections run fused_linear; larger batches go to the GEMM library with the fused operations around
# it. At 32 tokens (0.5B layer, us) 33 against 51; at 64, 46 against 56 with the gated projection alone slower, at 128
# 60 against 52.
MAX_TOKENS = 32
# From here on four workgroups share a row tile's K: 11.6 -> 7.0 us at 896 x 4864 and 8 tokens, 19.1 -> 12.9 at
# 1536 x 8960; at 896 x 896 the merge would cost more than the rows' whole read.
SPLIT_FEATURES = 4096


def _ok(t, device: torch.device, dim: int) -> bool:
    return (type(t) is torch.Tensor or type(t) is torch.nn.Parameter) and t.dtype == torch.bfloat16 and \
        t.device == device and t.dim() == dim and t.is_contiguous() and t.data_ptr() % 16 == 0


def rows_ok(x: torch.Tensor, norm_weight: torch.Tensor) -> bool:
    """Whether rms_norm can run on rows x [T, K]. Only under torch.inference_mode: the kernels record nothing for
    autograd, and forward-mode derivatives and saved-tensor hooks do not reach them there."""
    return torch.is_inference_mode_enabled() and x.is_cuda and _ok(x, x.device, 2) and x.shape[1] % 8 == 0 and \
        x.shape[1] <= 8192 and _ok(norm_weight, x.device, 1) and norm_weight.shape[0] == x.shape[1]


def supported(x: torch.Tensor, w, rot, heads: int, head_dim: int) -> bool:
    """Whether the layer w (engine.model.Layer) with `heads` query, key and value heads can run on hidden states
    x [T, hidden] with the kernels below: bf16, contiguous, 16-byte aligned tensors of one GPU whose sizes are whole
    tiles. The model's torch operations serve everything else, and raise their own errors for sizes that disagree."""
    if not (rows_ok(x, w.input_norm) and head_dim % 16 == 0):
        return False
    T, hidden = x.shape
    dev, width, inter = x.device, heads * head_dim, w.down_w.shape[-1]
    cos, sin = rot
    return (hidden % 64 == 0 and inter % 64 == 0 and w.o_w.shape[-1] % 64 == 0 and
            _ok(w.qkv_w, dev, 2) and tuple(w.qkv_w.shape) == (width, hidden) and
            _ok(w.qkv_b, dev, 1) and w.qkv_b.shape[0] == width and
            _ok(w.o_w, dev, 2) and w.o_w.shape[0] == hidden and
            _ok(w.post_norm, dev, 1) and w.post_norm.shape[0] == hidden and
            _ok(w.gate_up_w, dev, 2) and tuple(w.gate_up_w.shape) == (2 * inter, hidden) and
            _ok(w.down_w, dev, 2) and w.down_w.shape[0] == hidden and
            _ok(cos, dev, 3) and tuple(cos.shape) == (T, 1, head_dim) and
            _ok(sin, dev, 3) and tuple(sin.shape) == (T, 1, head_dim))


def fused_linear(x: torch.Tensor, weight: torch.Tensor, epilogue: int, *, norm_weight: torch.Tensor | None = None,
                 eps: float = 0.0, bias: torch.Tensor | None = None, residual: torch.Tensor | None = None,
                 rot: tuple[torch.Tensor, torch.Tensor] | None = None, head_dim: int = 0,
                 rot_channels: int = 0, num_splits: int = 1) -> torch.Tensor:
    """epilogue(norm(x) W^T) in one launch (sipa_fused_linear): x [T, K], weight [N, K]; RESIDUAL adds bias and
    residual, ROPE adds bias and rotates the first rot_channels channels by rot = (cos, signed sin), SILU multiplies
    the second half of the channels by silu of the first."""
    T, K = x.shape
    N = weight.shape[0]
    out = torch.empty(T, N // 2 if epilogue == SILU else N, device=x.device, dtype=torch.bfloat16)
    part = counters = None
    if num_splits > 1:
        groups = 1 if T <= 16 else 2 if T <= 32 else 4 * -(-T // 64)
        part = torch.empty(N // 16 * groups * num_splits * 256, device=x.device, dtype=torch.float32)
        counters = reserve_workspace(x.device, _hip.stream_of(x), 0)
    p = _hip.LinearParams(ctypes.sizeof(_hip.LinearParams), epilogue, T, K, N, head_dim, rot_channels, eps,
                          x.data_ptr(), x.stride(0), weight.data_ptr(), _hip.ptr(norm_weight), _hip.ptr(bias),
                          _hip.ptr(residual), residual.stride(0) if residual is not None else 0, out.data_ptr(),
                          out.stride(0), *((rot[0].data_ptr(), rot[1].data_ptr()) if rot is not None else (None, None)),
                          num_splits, _hip.ptr(part), _hip.ptr(counters))
    _hip.check(_hip.lib().sipa_fused_linear(ctypes.byref(p), _hip.stream_of(x)), "fused_linear")
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


def layer_qkv(x: torch.Tensor, w, eps: float, rot, rotated: int, head_dim: int) -> torch.Tensor:
    """[T, heads * head_dim]: the fused projection of the normalised x, its first `rotated` heads (queries and keys)
    rotated. One launch for a few tokens."""
    if x.shape[0] <= MAX_TOKENS:
        return fused_linear(x, w.qkv_w, ROPE, norm_weight=w.input_norm, eps=eps, bias=w.qkv_b, rot=rot,
                            head_dim=head_dim, rot_channels=rotated * head_dim)
    qkv = F.linear(rms_norm(x, w.input_norm, eps), w.qkv_w, w.qkv_b)
    rope_(qkv, rot, rotated, head_dim)
    return qkv


def layer_out(x: torch.Tensor, attn: torch.Tensor, w, eps: float) -> torch.Tensor:
    """x + attn W_o, then that plus its MLP. Three launches for a few tokens."""
    if x.shape[0] <= MAX_TOKENS:
        h = fused_linear(attn, w.o_w, RESIDUAL, residual=x)
        act = fused_linear(h, w.gate_up_w, SILU, norm_weight=w.post_norm, eps=eps)
        return fused_linear(act, w.down_w, RESIDUAL, residual=h,
                            num_splits=4 if w.down_w.shape[1] >= SPLIT_FEATURES else 1)
    n, h = rms_norm(x, w.post_norm, eps, add=F.linear(attn, w.o_w))
    return h + F.linear(silu_mul(F.linear(n, w.gate_up_w)), w.down_w)
