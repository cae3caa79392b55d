"""Ragged causal GQA paged prefill on gfx950 -- drop-in for
``vllm/kernels/prefill_paged_attention.py:prefill_paged_attention``.

Same positional arguments, keywords, shapes and ``ValueError`` checks as the
reference entry (prefill_paged_attention.py:391-453, checks :189-207,
:430-431).  Tensors are torch tensors on a HIP device; ``k_pages`` /
``v_pages`` are ``[Hkv, NB, BS, d]`` *views* -- any strides with a unit last
stride -- so the engine's native pool ``kv_cache[i]`` (``[NB, BS, Hkv, d]``)
is passed as ``kv_cache[i].permute(2, 0, 1, 3)`` without the full-pool
transpose the reference performs (qwen3.py:177-178).

The Pallas tuning knobs (``block_m``, ``block_h``, ``pages_per_compute_block``,
``k_splits``, ``num_warps``, ``num_stages``, ``interpret``, ``debug``) are
accepted and ignored.  ``mask_value`` only matters for rows with no visible
key, which this implementation returns as zeros.
"""
from __future__ import annotations

import torch

from .. import _lib
from ._common import (DEFAULT_MASK_VALUE, as_i32, check_quantized_pages, inv_sqrt_head_dim_bf16, pages_strides,
                      pool_pointers, require_bf16, require_device, stream_handle)

_ROUTE_SPLIT = 2  # PA_PREFILL_SPLIT


def prefill_paged_attention(
        q: torch.Tensor,
        k_pages: torch.Tensor,
        v_pages: torch.Tensor,
        block_tables: torch.Tensor,
        cu_seqlens: torch.Tensor,
        slot_mapping: torch.Tensor,
        input_positions: torch.Tensor,
        *,
        max_seqlen_bucket: int,
        k_scales_pages: torch.Tensor | None = None,
        v_scales_pages: torch.Tensor | None = None,
        block_m: int = 16,
        block_h: int = 16,
        pages_per_compute_block: int = 8,
        k_splits: int = 8,
        num_warps: int = 8,
        num_stages: int = 2,
        interpret: bool = False,
        debug: bool = False,
        mask_value: float = DEFAULT_MASK_VALUE,
        attn_logits_soft_cap: float | None = None,
        cu_seqlens_k: torch.Tensor | None = None,
        scale: float | None = None,
        out: torch.Tensor | None = None,
        workspace: torch.Tensor | None = None,
        max_seqlen_k: int | None = None,
) -> torch.Tensor:
    """Paged prefill attention; returns ``[T, H, d]`` bf16.

    Extensions beyond the reference signature (all keyword-only, defaulting
    to the reference behaviour):
      * ``cu_seqlens_k`` -- per-sequence kv lengths including a cached prefix;
        kv index j then sits at position ``j + pos0 - (Lk - Lq)``;
      * ``scale`` -- logit scale (default: bf16(1/sqrt(d)) as prefill...:60);
      * ``out`` -- preallocated output;
      * ``workspace`` -- device bytes for the work list that orders the
        kernel's items by kv length (``pa_prefill_workspace_size``; with
        ``pa_prefill_split_workspace_size`` bytes a launch of few, long items
        also splits them over their kv range, which changes the last bits of
        its results by the batch's lengths) and, for
        quantized pages (float8 e4m3fn codes, or int8 / uint8 integers, with
        float32 ``[Hkv, NB, BS]`` per-token scales), the pages widened to bf16 ahead of it
        (``pa_prefill_fp8_workspace_size``); allocated when absent or too small;
      * ``max_seqlen_k`` -- a bound on the kv lengths (0: none is known), where
        ``block_tables`` is wider than the longest of them: launches are split
        by the bound instead of the table's width.  It changes no result but
        the last bits of a launch that it keeps whole.
    """
    del slot_mapping, block_m, pages_per_compute_block, k_splits, num_warps, num_stages
    del interpret, debug, mask_value
    if block_h % 16:
        raise ValueError(f"block_h must divisible by 16, but is {block_h}.")
    if tuple(k_pages.shape) != tuple(v_pages.shape):
        raise ValueError(
            f"k_pages and v_pages must have the same shape. Got {tuple(k_pages.shape)} and"
            f" {tuple(v_pages.shape)}")
    _check_shapes(q, k_pages.shape, block_tables, cu_seqlens, cu_seqlens_k)
    code_type = check_quantized_pages(k_pages, v_pages, k_scales_pages, v_scales_pages)
    for name, t in (("k_pages", k_pages), ("v_pages", v_pages)):
        require_device(name, t)
        if code_type is None:
            require_bf16(name, t)
    if tuple(k_pages.stride()) != tuple(v_pages.stride()):
        raise ValueError("k_pages and v_pages must share strides")
    num_kv_heads, num_pages, page_size, head_dim = k_pages.shape
    scales = () if code_type is None else (k_scales_pages.data_ptr(), v_scales_pages.data_ptr(),
                                           k_scales_pages.stride(1), k_scales_pages.stride(0))
    return _prefill(q, (num_kv_heads, num_pages, page_size, head_dim), (k_pages.data_ptr(), v_pages.data_ptr()),
                    pages_strides(k_pages), code_type, scales, block_tables, cu_seqlens, input_positions,
                    max_seqlen_bucket, attn_logits_soft_cap, cu_seqlens_k, scale, out, workspace, max_seqlen_k)


def prefill_pool(q: torch.Tensor, kv_cache: torch.Tensor, block_tables: torch.Tensor, cu_seqlens: torch.Tensor,
                 input_positions: torch.Tensor, *, max_seqlen_bucket: int,
                 cu_seqlens_k: torch.Tensor | None = None, max_seqlen_k: int | None = None) -> torch.Tensor:
    """:func:`prefill_paged_attention` over the halves of the engine's bf16
    pool ``[2, NB, BS, Hkv, d]``, without making the page views."""
    require_device("kv_cache", kv_cache)
    require_bf16("kv_cache", kv_cache)
    _, num_pages, page_size, num_kv_heads, head_dim = kv_cache.shape
    _check_shapes(q, (num_kv_heads, num_pages, page_size, head_dim), block_tables, cu_seqlens, cu_seqlens_k)
    _, ps, ss, hs, _ = kv_cache.stride()
    return _prefill(q, (num_kv_heads, num_pages, page_size, head_dim), pool_pointers(kv_cache), (ps, ss, hs), None, (),
                    block_tables, cu_seqlens, input_positions, max_seqlen_bucket, None, cu_seqlens_k, None, None, None,
                    max_seqlen_k)


def _check_shapes(q, pages, block_tables, cu_seqlens, cu_seqlens_k):
    num_heads, head_dim = q.shape[1:]
    num_kv_heads, head_dim_k = pages[0], pages[3]
    batch = block_tables.shape[0]
    if num_heads % num_kv_heads != 0:
        raise ValueError(
            "Number of Q heads must be divisible by number of KV heads. Got"
            f" {num_heads} and {num_kv_heads}.")
    if head_dim_k != head_dim:
        raise ValueError(
            "head_dim of Q must be the same as that of K/V. Got"
            f" {head_dim} and {head_dim_k}.")
    if tuple(cu_seqlens.shape) != (batch + 1,):
        raise ValueError("cu_seqlens must have shape [batch + 1]")
    if block_tables.dtype != torch.int32:
        raise ValueError("block_tables must be int32")
    if cu_seqlens_k is not None and tuple(cu_seqlens_k.shape) != (batch + 1,):
        raise ValueError("cu_seqlens_k must have shape [batch + 1]")


def _prefill(q, pages, pointers, strides, code_type, scales, block_tables, cu_seqlens, input_positions,
             max_seqlen_bucket, attn_logits_soft_cap, cu_seqlens_k, scale, out, workspace, max_seqlen_k):
    """The launch for checked pages: ``pages`` = (Hkv, NB, BS, d), ``pointers``
    and element ``strides`` (page, slot, head) of K and V, ``scales`` =
    pointers and (page, head) strides of quantized pages' scales."""
    total_tokens, num_heads, head_dim = q.shape
    num_kv_heads, total_num_pages, page_size, _ = pages
    batch, pages_per_sequence = block_tables.shape
    for name, t in (("q", q), ("block_tables", block_tables), ("cu_seqlens", cu_seqlens),
                    ("input_positions", input_positions)):
        require_device(name, t)
    require_bf16("q", q)
    bt = block_tables if block_tables.stride(-1) == 1 else block_tables.contiguous()
    cu = as_i32("cu_seqlens", cu_seqlens)
    cuk = as_i32("cu_seqlens_k", cu_seqlens_k) if cu_seqlens_k is not None else None
    pos = as_i32("input_positions", input_positions)
    if out is None:
        out = torch.empty_like(q, memory_format=torch.contiguous_format)
    else:
        require_device("out", out)
        require_bf16("out", out)
        if tuple(out.shape) != tuple(q.shape):
            raise ValueError(f"out must have shape {tuple(q.shape)}")
    if scale is None:
        scale = inv_sqrt_head_dim_bf16(head_dim)
    soft_cap = 0.0 if attn_logits_soft_cap is None else float(attn_logits_soft_cap)
    ps, ss, hs = strides
    quantized = code_type is not None
    lib = _lib.load()
    need = int(lib.pa_prefill_workspace_size(batch, int(max_seqlen_bucket), num_heads, num_kv_heads))
    extra = 0  # bytes of the widened pages
    if quantized:
        extra = int(lib.pa_prefill_fp8_workspace_size(batch, pages_per_sequence, page_size, num_kv_heads, head_dim,
                                                      int(max_seqlen_bucket), num_heads)) - need
    given = 0 if workspace is None else workspace.numel() * workspace.element_size()
    if given < need + extra or max_seqlen_k is not None:
        pages = pages_per_sequence
        if max_seqlen_k is not None:
            pages = min(pages, -(-max(0, int(max_seqlen_k)) // page_size))
        cached = cuk is not None and cuk.data_ptr() != cu.data_ptr()
        split = lib.pa_prefill_route(batch, total_tokens, int(max_seqlen_bucket), num_heads, num_kv_heads, head_dim,
                                     pages, page_size, cached) == _ROUTE_SPLIT
        if given < need + extra:
            # our own: with room for the parts of a launch that splits its items
            if split:
                need = int(lib.pa_prefill_split_workspace_size(batch, int(max_seqlen_bucket), num_heads, num_kv_heads,
                                                               head_dim, pages_per_sequence, page_size))
            given = max(need + extra, 1)
            workspace = torch.empty(given, dtype=torch.uint8, device=q.device)
        elif not split:
            given = need + extra  # no room for parts
    if quantized:
        _lib.call(
            "pa_prefill_quant", code_type,
            q.data_ptr(), q.stride(0), q.stride(1),
            *pointers, scales[0], scales[1],
            total_num_pages, page_size, ps, ss, hs,
            scales[2], scales[3],
            bt.data_ptr(), bt.stride(0), pages_per_sequence,
            cu.data_ptr(), cuk.data_ptr() if cuk is not None else None, pos.data_ptr(),
            batch, total_tokens, int(max_seqlen_bucket),
            num_heads, num_kv_heads, head_dim,
            float(scale), soft_cap,
            out.data_ptr(), out.stride(0), out.stride(1),
            workspace.data_ptr(), given,
            stream_handle(q))
        return out
    _lib.call(
        "pa_prefill",
        q.data_ptr(), q.stride(0), q.stride(1),
        *pointers, total_num_pages, page_size,
        ps, ss, hs,
        bt.data_ptr(), bt.stride(0), pages_per_sequence,
        cu.data_ptr(), cuk.data_ptr() if cuk is not None else None, pos.data_ptr(),
        batch, total_tokens, int(max_seqlen_bucket),
        num_heads, num_kv_heads, head_dim,
        float(scale), soft_cap,
        out.data_ptr(), out.stride(0), out.stride(1),
        workspace.data_ptr(), given,
        stream_handle(q))
    return out
