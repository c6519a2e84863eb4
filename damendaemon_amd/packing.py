"""GPU ragged-batch packer and K/V page writer.

``pack_batch`` replaces the host-side packing of damendaemon/paged.py:149-159
(flat ``positions``/``slot_ids`` built by list comprehensions), the
``accumulate(lengths)`` segment ends of paged.py:118-120 and the physical
slot computation of kernels.py:279-281: the (length, start, slot) of every
segment travel in the launch's arguments and the GPU expands them.
"""
from dataclasses import dataclass

import numpy as np
import torch

from . import _native
from ._native import call, ptr


@dataclass
class PackedBatch:
    """Device outputs of ``pack_batch`` (int64 unless noted) plus host sizes."""
    cu_seqlens: torch.Tensor      # (n+1,)
    ends: torch.Tensor            # (n,)  last token of each segment
    context_lens: torch.Tensor    # (n,)  start + length
    positions: torch.Tensor       # (T,)
    slot_ids: torch.Tensor        # (T,)
    slot_map: torch.Tensor        # (T,)  physical page * P + offset, or None
    cu_pages: torch.Tensor        # (n+1,) int32, or None
    gather_pages: torch.Tensor    # (total_pages,) int32, or None
    lengths: list
    starts: list
    slots: list
    total_tokens: int
    page_size: int


def pack_batch(lengths, starts, slots, page_table=None, page_size=16, device='cuda', gather=True):
    """Pack n segments (len_i tokens appended after start_i cached tokens of slot_i).

    ``lengths``, ``starts`` and ``slots`` are host integer sequences (the
    scheduler's own lists).  With a ``page_table`` the slot map and the page
    gather lists are produced too.
    """
    try:
        host = np.array((lengths, starts, slots), dtype=np.int64)
    except (TypeError, ValueError, OverflowError):
        raise ValueError('invalid packing request') from None
    if host.ndim != 2 or page_size <= 0 or (host[:2] < 0).any():
        raise ValueError('invalid packing request')
    n = host.shape[1]
    lengths, starts, slots = host.tolist()
    total = sum(lengths)
    with_table = page_table is not None
    gather = gather and with_table
    pages = sum([(a + b + (page_size - 1)) // page_size for a, b in zip(lengths, starts)]) if gather else 0
    dev = torch.device(device)
    if dev.type != 'cuda':
        raise ValueError('damendaemon_amd kernels need tensors on the GPU (there is no CPU path)')
    _native.refuse_capture()
    _native.require_device(page_table)
    if with_table and (page_table.dtype != torch.int32 or not page_table.is_contiguous()):
        raise ValueError('page table must be a contiguous int32 matrix')
    # one allocation for the int64 outputs and one for the int32 ones
    sizes = [n + 1, n, n, 3 * n, total, total, total if with_table else 0]
    buffer = torch.empty(sum(sizes), dtype=torch.int64, device=dev)
    cu_seqlens, ends, context_lens, meta, positions, slot_ids, slot_map = buffer.split(sizes)
    cu_pages, gather_pages = (torch.empty(n + 1 + pages, dtype=torch.int32, device=dev).split([n + 1, pages])
                              if gather else (None, None))
    meta = meta.view(3, n)
    out = PackedBatch(cu_seqlens, ends, context_lens, positions, slot_ids, slot_map if with_table else None, cu_pages,
                      gather_pages, lengths, starts, slots, total, page_size)
    table_args = (ptr(page_table), *(page_table.shape if with_table else (0, 0)), page_size)
    results = (ptr(positions), ptr(slot_ids), ptr(out.slot_map), ptr(cu_pages), ptr(gather_pages),
               _native.stream_of(buffer))
    source = host.ctypes.data
    code = _native.UNSUPPORTED
    if n:
        code = _native.status('dd_pack_batch_host', source, source + 8 * n, source + 16 * n, n, total, pages, *table_args,
                              ptr(cu_seqlens), ptr(ends), ptr(context_lens), ptr(meta), *results)
    if code == _native.UNSUPPORTED:   # no segments, or values past 30 bits
        meta.copy_(_native.upload(torch.from_numpy(host), buffer.device))
        first = ptr(meta)
        call('dd_pack_batch', first, first + 8 * n, first + 16 * n, n, total, pages, *table_args, ptr(cu_seqlens),
             ptr(ends), ptr(context_lens), *results)
    elif code:
        _native.check('dd_pack_batch_host', code)
    out._meta, out._host = meta, host
    return out


def store_kv_pages(key, value, slot_map, cache_k, cache_v, k_scale=None, v_scale=None):
    """Write (T, KH, D) keys/values into their page slots.

    bf16/fp16/fp32 caches take the rows as they are (cast to the cache dtype
    first); int8 caches (with fp16 ``k_scale``/``v_scale`` (..., page, D/group))
    quantise each row group to Q8_0 on the way in.
    """
    tokens, kv_heads, dim = key.shape
    capacity, kvh, page, cdim = cache_k.shape
    if (value.shape != key.shape or kvh != kv_heads or cdim != dim or slot_map.shape != (tokens,)
            or cache_v.shape != cache_k.shape or not cache_k.is_contiguous() or not cache_v.is_contiguous()):
        raise ValueError('incompatible K/V page write shapes')
    _native.require_device(key, value, slot_map, cache_k, cache_v)
    if slot_map.dtype != torch.int64:
        slot_map = slot_map.to(torch.int64)
    if cache_k.dtype == torch.int8:
        if k_scale is None or v_scale is None or k_scale.shape[:-1] != cache_k.shape[:-1] or dim % k_scale.shape[-1]:
            raise ValueError('int8 pages need fp16 scales (..., page, dim/group)')
        key, value = key.contiguous(), value.contiguous()
        call('dd_store_kv_pages_q8', ptr(key), ptr(value), _native.DTYPE_CODES[key.dtype], ptr(slot_map), tokens,
             kv_heads, dim, dim // k_scale.shape[-1], page, capacity, ptr(cache_k), ptr(cache_v), ptr(k_scale),
             ptr(v_scale), _native.stream_of(key))
        return
    key = key.to(cache_k.dtype).contiguous()
    value = value.to(cache_k.dtype).contiguous()
    call('dd_store_kv_pages', ptr(key), ptr(value), cache_k.element_size(), ptr(slot_map), tokens, kv_heads, dim,
         page, capacity, ptr(cache_k), ptr(cache_v), _native.stream_of(key))
