"""Fused INT8 quantize-and-store and plain scatter-store on MI355X through libsmallinf_hip.so: the drop-in for the
reference's engine/triton_quant.py (quantize_store_tokens, quantize_store_blocks; reference :61-84), plus the two
stores the reference leaves to torch ops (the pool scatter of engine/paged_cache.py:135-139 and format B's
staging and whole-block writes, engine/quant_cache.py:165-177).

The quantizer is bit-exact with engine/quant.py: scale = fp16(absmax / 127), code = clamp(rint(x / scale),
-127, 127) with IEEE fp32 division and round-half-even; a zero scale gives zero codes.
"""

from __future__ import annotations

import ctypes

import torch

from . import _hip


def _i64(t: torch.Tensor) -> torch.Tensor:
    """Index vectors go to the kernels as contiguous int64."""
    return t if (t.dtype == torch.int64 and t.is_contiguous()) else t.to(torch.int64).contiguous()


def _require(ok: bool, msg) -> None:
    """The kernels index the pools with the shapes given here: a mismatch is refused before any launch. msg: a text, or
    a function that makes it (formatted only when it is needed)."""
    if not ok:
        raise ValueError(msg if isinstance(msg, str) else msg())


def _token_pools(x: torch.Tensor, q_pool: torch.Tensor, s_pool: torch.Tensor) -> None:
    T, H, D = x.shape
    _require(q_pool.dim() == 4 and q_pool.shape[0] == H and q_pool.shape[3] == D,
             lambda: f"q_pool {tuple(q_pool.shape)} must be [H={H}, N, B, D={D}]")
    _require(tuple(s_pool.shape) == tuple(q_pool.shape[:3]),
             lambda: f"s_pool {tuple(s_pool.shape)} must be [H, N, B] = {tuple(q_pool.shape[:3])}")
    _require(q_pool.dtype == torch.int8 and s_pool.dtype == torch.float16, "q_pool must be int8 and s_pool fp16")
    _require(q_pool.is_contiguous() and s_pool.is_contiguous(), "the pools must be contiguous")


def quantize_store_tokens(x: torch.Tensor, blocks: torch.Tensor, offsets: torch.Tensor, q_pool: torch.Tensor,
                          s_pool: torch.Tensor, *, x2: torch.Tensor | None = None, q_pool2: torch.Tensor | None = None,
                          s_pool2: torch.Tensor | None = None) -> None:
    """x [T, H, D] (rows may be strided; last dim contiguous) -> q_pool [H, N, B, D] int8 and s_pool [H, N, B]
    fp16 at (blocks[t], offsets[t]). With x2, q_pool2, s_pool2 (the other of K and V, same shapes) both pairs are
    stored in the same launch, equal bit for bit to two calls. One launch."""
    T, H, D = x.shape
    if T == 0:
        return
    _require(x.stride(-1) == 1, "x needs a contiguous last dim")
    _require(blocks.numel() == T and offsets.numel() == T, lambda: f"{T} tokens need {T} blocks and offsets")
    _token_pools(x, q_pool, s_pool)
    _hip.require_gpu(x, blocks, offsets, q_pool, s_pool)
    blocks, offsets = _i64(blocks), _i64(offsets)
    if x2 is not None:
        if q_pool2 is None or s_pool2 is None:
            raise ValueError("x2 needs q_pool2 and s_pool2")
        if x2.shape != x.shape or x2.dtype != x.dtype or x2.stride(-1) != 1:
            raise ValueError("x2 must match x in shape and dtype, last dim contiguous")
        if (q_pool2.shape, q_pool2.stride(), q_pool2.dtype) != (q_pool.shape, q_pool.stride(), q_pool.dtype) or \
                (s_pool2.shape, s_pool2.stride(), s_pool2.dtype) != (s_pool.shape, s_pool.stride(), s_pool.dtype):
            raise ValueError("the second pools must match the first in shape, strides and dtype")
        _hip.require_gpu(x2, q_pool2, s_pool2)
        rc = _hip.lib().sipa_quantize_store_tokens_kv(
            x.data_ptr(), x2.data_ptr(), _hip.dtype_code(x.dtype), x.stride(0), x.stride(1), x2.stride(0),
            x2.stride(1), T, H, D, blocks.data_ptr(), offsets.data_ptr(), q_pool.data_ptr(), q_pool2.data_ptr(),
            q_pool.stride(0), q_pool.stride(1), q_pool.shape[2], s_pool.data_ptr(), s_pool2.data_ptr(),
            s_pool.stride(0), s_pool.stride(1), _hip.stream_of(x))
        _hip.check(rc, "quantize_store_tokens")
        return
    rc = _hip.lib().sipa_quantize_store_tokens(
        x.data_ptr(), _hip.dtype_code(x.dtype), x.stride(0), x.stride(1), T, H, D, blocks.data_ptr(),
        offsets.data_ptr(), q_pool.data_ptr(), q_pool.stride(0), q_pool.stride(1), q_pool.shape[2],
        s_pool.data_ptr(), s_pool.stride(0), s_pool.stride(1), _hip.stream_of(x))
    _hip.check(rc, "quantize_store_tokens")


def quantize_store_blocks(src_pool: torch.Tensor, src: torch.Tensor, dst: torch.Tensor, q_pool: torch.Tensor,
                          s_pool: torch.Tensor) -> None:
    """Blocks src_pool[:, src[i]] ([H, n_src, B, D], e.g. bf16 staging) -> q_pool[:, dst[i]] int8 with per-channel
    scales s_pool[:, dst[i]] ([H, N, D] fp16). One launch."""
    if src.numel() == 0:
        return
    H, _, B, D = src_pool.shape
    _require(src.numel() == dst.numel(), lambda: f"{src.numel()} sources for {dst.numel()} destinations")
    _require(q_pool.dim() == 4 and (q_pool.shape[0], q_pool.shape[2], q_pool.shape[3]) == (H, B, D),
             lambda: f"q_pool {tuple(q_pool.shape)} must be [H={H}, N, B={B}, D={D}]")
    _require(tuple(s_pool.shape) == (H, q_pool.shape[1], D), lambda: f"s_pool {tuple(s_pool.shape)} must be [H, N, D]")
    _require(q_pool.dtype == torch.int8 and s_pool.dtype == torch.float16, "q_pool must be int8 and s_pool fp16")
    _require(src_pool.is_contiguous() and q_pool.is_contiguous() and s_pool.is_contiguous(),
             "the pools must be contiguous")
    _hip.require_gpu(src_pool, src, dst, q_pool, s_pool)
    src, dst = _i64(src), _i64(dst)
    rc = _hip.lib().sipa_quantize_store_blocks(
        src_pool.data_ptr(), _hip.dtype_code(src_pool.dtype), src_pool.stride(0), src_pool.stride(1),
        src_pool.stride(2), src.data_ptr(), dst.data_ptr(), src.numel(), H, B, D, q_pool.data_ptr(),
        q_pool.stride(0), q_pool.stride(1), s_pool.data_ptr(), s_pool.stride(0), s_pool.stride(1),
        _hip.stream_of(src_pool))
    _hip.check(rc, "quantize_store_blocks")


def quantize_store_block_rows(x: torch.Tensor, rows: torch.Tensor, dst: torch.Tensor, q_pool: torch.Tensor,
                              s_pool: torch.Tensor) -> None:
    """Whole blocks taken from rows of x [T, H, D]: block i is rows[i*B : (i+1)*B] (B = q_pool's block size),
    rounded to bf16, then quantized per channel into q_pool[:, dst[i]], s_pool[:, dst[i]]. One launch."""
    if dst.numel() == 0:
        return
    H, _, B, D = q_pool.shape
    _require(x.dim() == 3 and x.shape[1] == H and x.shape[2] == D and x.stride(-1) == 1,
             lambda: f"x {tuple(x.shape)} must be [T, H={H}, D={D}] with a contiguous last dim")
    _require(tuple(s_pool.shape) == (H, q_pool.shape[1], D), lambda: f"s_pool {tuple(s_pool.shape)} must be [H, N, D]")
    _require(q_pool.dtype == torch.int8 and s_pool.dtype == torch.float16, "q_pool must be int8 and s_pool fp16")
    _require(q_pool.is_contiguous() and s_pool.is_contiguous(), "the pools must be contiguous")
    _require(rows.numel() == dst.numel() * B, lambda: f"{rows.numel()} rows for {dst.numel()} blocks of {B}")
    _hip.require_gpu(x, rows, dst, q_pool, s_pool)
    rows, dst = _i64(rows), _i64(dst)
    rc = _hip.lib().sipa_quantize_store_block_rows(
        x.data_ptr(), _hip.dtype_code(x.dtype), x.stride(0), x.stride(1), rows.data_ptr(), dst.data_ptr(),
        dst.numel(), H, B, D, q_pool.data_ptr(), q_pool.stride(0), q_pool.stride(1), s_pool.data_ptr(),
        s_pool.stride(0), s_pool.stride(1), _hip.stream_of(x))
    _hip.check(rc, "quantize_store_block_rows")


def store_tokens(x: torch.Tensor, blocks: torch.Tensor, offsets: torch.Tensor, pool: torch.Tensor,
                 rows: torch.Tensor | None = None, x2: torch.Tensor | None = None,
                 pool2: torch.Tensor | None = None) -> None:
    """pool[:, blocks[i], offsets[i]] = x[rows[i] if rows is not None else i] (x [T, H, D], pool [H, N, B, D]),
    converted to the pool's dtype with round-to-nearest-even; (x2, pool2) in the same launch (x2 may have other
    strides than x, as K and V views of a fused projection do). One launch."""
    n = blocks.numel()
    if n == 0:
        return
    T, H, D = x.shape
    _require(x.stride(-1) == 1 and pool.stride(-1) == 1, "x and the pool need a contiguous last dim")
    _require(pool.dim() == 4 and pool.shape[0] == H and pool.shape[3] == D,
             lambda: f"pool {tuple(pool.shape)} must be [H={H}, N, B, D={D}]")
    _require(offsets.numel() == n, lambda: f"{n} blocks but {offsets.numel()} offsets")
    _require(n <= T if rows is None else rows.numel() == n, "one source row per stored token")
    if x2 is not None:
        _require(x2.shape == x.shape and x2.stride(-1) == 1 and x2.dtype == x.dtype,
                 "x2 must match x in shape and dtype, last dim contiguous")
        _require(pool2 is not None and pool2.shape == pool.shape and pool2.stride() == pool.stride() and
                 pool2.dtype == pool.dtype, "pool2 must match the pool in shape, strides and dtype")
        _hip.require_gpu(x2, pool2)
    _hip.require_gpu(x, blocks, offsets, pool)
    blocks, offsets = _i64(blocks), _i64(offsets)
    rows = None if rows is None else _i64(rows)
    rc = _hip.lib().sipa_store_tokens(
        x.data_ptr(), _hip.ptr(x2), _hip.dtype_code(x.dtype), x.stride(0), x.stride(1),
        x.stride(0) if x2 is None else x2.stride(0), x.stride(1) if x2 is None else x2.stride(1), _hip.ptr(rows), n, H, D,
        blocks.data_ptr(), offsets.data_ptr(), pool.data_ptr(), _hip.ptr(pool2), _hip.dtype_code(pool.dtype),
        pool.stride(0), pool.stride(1), pool.stride(2), _hip.stream_of(x))
    _hip.check(rc, "store_tokens")


def _kv_rows(k: torch.Tensor, v: torch.Tensor, blocks: torch.Tensor, offsets: torch.Tensor, k_pools: torch.Tensor,
             v_pools: torch.Tensor, need_all: bool) -> None:
    """Checks that store_layer and quantize_store_layer share: K and V rows [T, H, D], their slots (for every row, or for
    the first ones), and pools [L, H, N, B, D]."""
    rows, shape, n = k.shape, k_pools.shape, blocks.numel()
    if v.shape != rows or v.dtype != k.dtype or k.stride(-1) != 1 or v.stride(-1) != 1:
        raise ValueError("k and v must match in shape and dtype, last dim contiguous")
    if offsets.numel() != n or n > rows[0] or need_all and n < rows[0]:
        raise ValueError(f"{n} blocks and {offsets.numel()} offsets for {rows[0]} rows")
    if len(shape) != 5 or shape[1] != rows[1] or shape[4] != rows[2] or v_pools.shape != shape:
        raise ValueError(f"pools {tuple(shape)} and {tuple(v_pools.shape)} must both be [L, H={rows[1]}, N, B, D={rows[2]}]")


def store_layer(layer: int, k: torch.Tensor, v: torch.Tensor, blocks: torch.Tensor, offsets: torch.Tensor,
                k_pools: torch.Tensor, v_pools: torch.Tensor) -> None:
    """store_tokens(k, blocks, offsets, k_pools[layer], x2=v, pool2=v_pools[layer]) for pools [L, H, N, B, D], without
    making the layer's views. One launch."""
    n = blocks.numel()
    if n == 0:
        return
    strides = k_pools.stride()
    _kv_rows(k, v, blocks, offsets, k_pools, v_pools, False)
    _require(strides[4] == 1 and v_pools.stride()[1:] == strides[1:] and v_pools.dtype == k_pools.dtype,
             "the pools must match in strides and dtype, last dim contiguous")
    _hip.require_gpu(k, v, blocks, offsets, k_pools, v_pools)
    blocks, offsets = _i64(blocks), _i64(offsets)
    (kt, kh, _), (vt, vh, _) = k.stride(), v.stride()
    rc = _hip.lib().sipa_store_tokens(
        k.data_ptr(), v.data_ptr(), _hip.dtype_code(k.dtype), kt, kh, vt, vh, None, n, *k.shape[1:], blocks.data_ptr(),
        offsets.data_ptr(), _hip.layer_ptr(k_pools, layer), _hip.layer_ptr(v_pools, layer),
        _hip.dtype_code(k_pools.dtype), strides[1], strides[2], strides[3], _hip.stream_of(k))
    if rc:
        _hip.check(rc, "store_tokens")


def quantize_store_layer(layer: int, k: torch.Tensor, v: torch.Tensor, blocks: torch.Tensor, offsets: torch.Tensor,
                         k_pools: torch.Tensor, k_scales: torch.Tensor, v_pools: torch.Tensor,
                         v_scales: torch.Tensor) -> None:
    """quantize_store_tokens of v and k into layer `layer` of pools [L, H, N, B, D] and scales [L, H, N, B], without
    making the layer's views. One launch."""
    T, H, D = k.shape
    if T == 0:
        return
    _kv_rows(k, v, blocks, offsets, k_pools, v_pools, True)
    shape = k_pools.shape
    if k_scales.shape != shape[:4] or v_scales.shape != shape[:4]:
        raise ValueError(f"scales must be [L, H, N, B] = {tuple(shape[:4])}")
    if k_pools.dtype is not torch.int8 or v_pools.dtype is not torch.int8 or \
            k_scales.dtype is not torch.float16 or v_scales.dtype is not torch.float16:
        raise ValueError("pools must be int8 and scales fp16")
    for t in (k_pools, v_pools, k_scales, v_scales):
        if not (t.is_contiguous() or _hip.layers_contiguous(t)):
            raise ValueError("the pools must be contiguous")
    _hip.require_gpu(k, v, blocks, offsets, k_pools, v_pools, k_scales, v_scales)
    blocks, offsets = _i64(blocks), _i64(offsets)
    (kt, kh, _), (vt, vh, _) = k.stride(), v.stride()
    _, qh, qn, _, _ = k_pools.stride()
    _, sh, sn, _ = k_scales.stride()
    rc = _hip.lib().sipa_quantize_store_tokens_kv(
        v.data_ptr(), k.data_ptr(), _hip.dtype_code(v.dtype), vt, vh, kt, kh, T, H, D, blocks.data_ptr(),
        offsets.data_ptr(), _hip.layer_ptr(v_pools, layer), _hip.layer_ptr(k_pools, layer), qh, qn, shape[3],
        _hip.layer_ptr(v_scales, layer), _hip.layer_ptr(k_scales, layer), sh, sn, _hip.stream_of(v))
    if rc:
        _hip.check(rc, "quantize_store_tokens")


def kchan_write_rows(k: torch.Tensor, v: torch.Tensor, blocks: torch.Tensor, offsets: torch.Tensor,
                     stage_slots: torch.Tensor, quant_dst: torch.Tensor | None, v_pool: torch.Tensor,
                     v_scale: torch.Tensor, k_pool: torch.Tensor, k_scale: torch.Tensor, stage: torch.Tensor) -> None:
    """Format B's writes of a decode step in one launch (no reference counterpart; the reference's cache makes
    three calls, engine/quant_cache.py:161-170): row t's V quantized per token at (blocks[t], offsets[t]), its K
    rounded to bf16 into stage[:, stage_slots[t], offsets[t]], and, when quant_dst[t] >= 0 (quant_dst None: when
    offsets[t] is the block's last offset, into blocks[t]), the slot's block quantized per channel into
    k_pool / k_scale. Equal bit for bit to quantize_store_tokens + store_tokens + quantize_store_blocks when no
    two rows share a staging slot."""
    T, H, D = v.shape
    if T == 0:
        return
    _require(k.shape == v.shape and k.dtype == v.dtype, "k and v must match in shape and dtype")
    _require(k.stride(-1) == 1 and v.stride(-1) == 1, "k and v need a contiguous last dim")
    _require(blocks.numel() == T and offsets.numel() == T and stage_slots.numel() == T,
             lambda: f"{T} rows need {T} blocks, offsets and staging slots")
    _require(quant_dst is None or quant_dst.numel() == T, lambda: f"quant_dst needs {T} entries")
    _token_pools(v, v_pool, v_scale)
    N, B = v_pool.shape[1], v_pool.shape[2]
    _require(tuple(k_pool.shape) == tuple(v_pool.shape) and k_pool.dtype == torch.int8 and k_pool.is_contiguous(),
             lambda: f"k_pool {tuple(k_pool.shape)} must be int8 {tuple(v_pool.shape)}, contiguous")
    _require(tuple(k_scale.shape) == (H, N, D) and k_scale.dtype == torch.float16 and k_scale.is_contiguous(),
             lambda: f"k_scale {tuple(k_scale.shape)} must be fp16 [H={H}, N={N}, D={D}], contiguous")
    _require(stage.dim() == 4 and (stage.shape[0], stage.shape[2], stage.shape[3]) == (H, B, D)
             and stage.dtype == torch.bfloat16 and stage.stride(-1) == 1,
             lambda: f"stage {tuple(stage.shape)} must be bf16 [H={H}, n_stage, B={B}, D={D}]")
    _hip.require_gpu(k, v, blocks, offsets, stage_slots, v_pool, v_scale, k_pool, k_scale, stage)
    blocks, offsets, stage_slots = _i64(blocks), _i64(offsets), _i64(stage_slots)
    if quant_dst is not None:
        _hip.require_gpu(quant_dst)
        quant_dst = _i64(quant_dst)
    p = _hip.KchanWriteParams()
    p.k, p.v, p.x_dtype = k.data_ptr(), v.data_ptr(), _hip.dtype_code(v.dtype)
    p.k_stride_t, p.k_stride_h, p.v_stride_t, p.v_stride_h = k.stride(0), k.stride(1), v.stride(0), v.stride(1)
    p.T, p.H, p.D, p.B = T, H, D, B
    p.blocks, p.offsets, p.stage_slots = blocks.data_ptr(), offsets.data_ptr(), stage_slots.data_ptr()
    p.quant_dst = quant_dst.data_ptr() if quant_dst is not None else None
    p.v_pool, p.v_scale, p.k_pool, p.k_scale = v_pool.data_ptr(), v_scale.data_ptr(), k_pool.data_ptr(), k_scale.data_ptr()
    p.q_stride_h, p.q_stride_n = v_pool.stride(0), v_pool.stride(1)
    p.vs_stride_h, p.vs_stride_n = v_scale.stride(0), v_scale.stride(1)
    p.ks_stride_h, p.ks_stride_n = k_scale.stride(0), k_scale.stride(1)
    p.stage, p.st_stride_h, p.st_stride_n, p.st_stride_b = stage.data_ptr(), stage.stride(0), stage.stride(1), stage.stride(2)
    _hip.check(_hip.lib().sipa_kchan_write_rows(ctypes.byref(p), _hip.stream_of(v)), "kchan_write_rows")
