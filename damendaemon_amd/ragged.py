"""Attention over one packed continuous batch: chunked prefill + decode rows.

The reference runs a prefill chunk as copy_pages (gather start+len tokens
into a dense tensor, damendaemon/paged.py:101-104) followed by torch SDPA
with a lower-right causal mask (qwen2.py:756-770), and decodes through
``kernels.attention`` in a separate forward pass (scheduler.py:822-873).
Here one packed token buffer (from ``packing.pack_batch``) is attended in
place: multi-token segments by the paged MFMA prefill kernel, the trailing
run of single-token segments by the split-KV decode kernel, one after the
other.  Both read the pages directly; nothing is gathered.
"""
import ctypes
import math
import os

import numpy as np
import torch

from . import _native, kernels
from ._native import DTYPE_CODES, call, ptr


def _check(query, cache_k, cache_v, page_table):
    if query.ndim == 4:
        query = query.reshape(query.shape[0], query.shape[1], query.shape[3])
    T, H, D = query.shape
    capacity, KH, page, kd = cache_k.shape
    if (kd != D or cache_v.shape != cache_k.shape or H % KH or cache_k.dtype != query.dtype
            or cache_v.dtype != query.dtype or query.dtype not in (torch.bfloat16, torch.float16, torch.float32)):
        raise ValueError('prefill attention needs bf16/fp16/fp32 query and pages of one dtype and head size')
    if not (query.is_contiguous() and cache_k.is_contiguous() and cache_v.is_contiguous()):
        raise ValueError('prefill attention needs contiguous tensors')
    if page_table.dtype != torch.int32 or page_table.ndim != 2 or not page_table.is_contiguous():
        raise ValueError('page table must be a contiguous int32 matrix')
    _native.require_device(query, cache_k, cache_v, page_table)
    return query


def prefill_plan(lengths, starts, heads, kv_heads, dim, window=0, slots=None, workgroups=0):
    """Schedule of the prefill kernel for these segments: a host int32 array
    (entries, 8), each row (item or -1, first packed token, length, start,
    slot, rounds, 0, 0); entry r * G + b is round r of workgroup b.

    Balances (segment, KV head, query tile) items over the XCDs, longest
    first, from the host copies of the segment lengths, starts and slots
    (slots default to 0 .. n-1).  ``workgroups`` > 0 (the number of CUs)
    gives each of at most that many workgroups a list of items to run in
    turn; 0 gives one item per workgroup.
    """
    lengths = np.ascontiguousarray(lengths, dtype=np.int64)
    starts = np.ascontiguousarray(starts, dtype=np.int64)
    slots = np.ascontiguousarray(np.arange(len(lengths)) if slots is None else slots, dtype=np.int64)
    if lengths.shape != starts.shape or lengths.shape != slots.shape or lengths.ndim != 1:
        raise ValueError('lengths, starts and slots must be matching 1-D sequences')
    lib = _native.library()
    args = (lengths.ctypes.data, starts.ctypes.data, slots.ctypes.data, len(lengths), heads, kv_heads, dim, int(window or 0),
            int(workgroups))
    # (a guess that holds for balanced schedules first: the length is only known once the schedule is)
    rows = 512 + 2 * kv_heads * int((lengths // 32 + 1).sum()) if workgroups > 0 else 0
    while True:
        plan = np.empty((max(rows, 1), PLAN_INTS), dtype=np.int32)
        need = lib.dd_prefill_plan(*args, plan.ctypes.data, rows)
        if need < 0:
            raise _native.NativeError(f'dd_prefill_plan failed: {lib.dd_error_string(-need).decode()} ({-need})')
        if need <= rows:
            return plan[:need]
        rows = need


PLAN_INTS = 8   # DD_PREFILL_PLAN_INTS


def prefill_split(lengths, starts, heads, kv_heads, dim, dtype, window, device):
    """(split_tiles, max_splits, scratch floats) of a prefill call on ``device``
    (dd_prefill_split), or None: a 16-bit call with more work items than CUs,
    or no kernel that splits."""
    lengths = np.ascontiguousarray(lengths, dtype=np.int64)
    starts = np.ascontiguousarray(starts, dtype=np.int64)
    tiles, splits, floats = ctypes.c_int(0), ctypes.c_int(1), ctypes.c_int64(0)
    code = _native.status('dd_prefill_split', lengths.ctypes.data, starts.ctypes.data, len(lengths), heads, kv_heads, dim,
                          DTYPE_CODES[dtype], int(window or 0), _cu_count(device), ctypes.byref(tiles),
                          ctypes.byref(splits), ctypes.byref(floats))
    return None if code else (tiles.value, splits.value, floats.value)


def prefill_attention(query, cache_k, cache_v, packed, page_table, window=0, scale=None, out=None,
                      segments=None, flags=None):
    """Causal attention of every packed query token over its slot's pages.

    query (T, H, D) or (T, H, 1, D); ``packed`` from ``pack_batch``; the
    chunk's own K/V must already be in the pages.  ``segments`` (a, b)
    restricts the work to segments a..b-1 (their tokens only).  ``flags``
    (optional, int32 on the device, at least ``prefill_flag_count`` entries)
    receives the bf16 kernel's per-item re-run flags; by default the call
    allocates them.
    """
    return prepare_prefill(query, cache_k, cache_v, packed, page_table, window, scale, out, segments, flags).run()


def prepare_prefill(query, cache_k, cache_v, packed, page_table, window=0, scale=None, out=None, segments=None,
                    flags=None):
    """Validate a prefill call, size its workspaces, upload its workgroup plan
    when it has more work items than the GPU has CUs, and return a
    ``PrefillLaunch`` whose ``run()`` only enqueues the kernels
    (arguments and errors as ``prefill_attention``)."""
    return _prepare_prefill(_check(query, cache_k, cache_v, page_table), cache_k, cache_v, packed, page_table, window,
                            scale, out, segments, flags)


def _prepare_prefill(q, cache_k, cache_v, packed, page_table, window, scale, out, segments, flags):
    T, H, D = q.shape
    capacity, KH, page, _ = cache_k.shape
    scale = float(D ** -.5 if scale is None else scale)
    if not math.isfinite(scale):
        raise ValueError('prefill attention needs a finite scale')
    if out is None:
        out = torch.empty_like(q)
    else:
        if (out.dtype != q.dtype or out.device != q.device or out.numel() != q.numel()
                or not out.is_contiguous()):
            raise ValueError('out must be a contiguous tensor of the query dtype, device and size')
        out = out.view(q.shape)
    count = len(packed.lengths)
    a, b = segments if segments is not None else (0, count)
    a, b, _ = slice(a, b).indices(count)
    if b <= a:
        return PrefillLaunch(out, None)
    n, window, code = b - a, int(window or 0), DTYPE_CODES[q.dtype]
    host = getattr(packed, '_host', None)
    if host is None:
        host = np.array((packed.lengths, packed.starts, packed.slots), dtype=np.int64)
    first = host.ctypes.data + 8 * a
    sizes = (ctypes.c_int64 * 7)()
    call('dd_prefill_prepare', first, first + 8 * count, n, H, KH, D, code, window, scale, _cu_count(q.device), sizes)
    schedule, split_tiles, max_splits, floats, n_flags, max_len, max_context = sizes
    if schedule:
        _native.refuse_capture()
    plan_dev, plan_len = None, 0
    if schedule == 2:
        # more work items than CUs: the MFMA kernel's XCD-balanced workgroup
        # order (with fewer there is nothing to order, and nothing to upload)
        plan = prefill_plan(host[0, a:b], host[1, a:b], H, KH, D, window, host[2, a:b],
                            _persistent_workgroups(q.device, D))
        if len(plan) == 0:
            return PrefillLaunch(out, None)
        plan_dev = _native.upload(torch.from_numpy(plan), q.device)
        plan_len = len(plan) // int(plan[0, 5])     # workgroups
    scratch = torch.empty(floats, dtype=torch.float32, device=q.device) if floats else None
    # per-item exactness flags of the bf16 kernel (written by the kernel itself)
    if flags is not None:
        if flags.dtype != torch.int32 or flags.device != q.device or flags.numel() < n_flags:
            raise ValueError(f'flags must be int32 on the query device with at least {n_flags} entries')
    elif n_flags:
        flags = torch.empty(n_flags, dtype=torch.int32, device=q.device)
    args = (q.data_ptr(), cache_k.data_ptr(), cache_v.data_ptr(), code, packed.cu_seqlens.data_ptr() + 8 * a,
            packed.context_lens.data_ptr() + 8 * a, packed._meta.data_ptr() + 8 * (2 * count + a), n, max_len,
            max_context, page_table.data_ptr(), *page_table.shape, H, KH, D, page, capacity, window, scale,
            ptr(plan_dev), plan_len, ptr(flags), out.data_ptr(), split_tiles, max_splits, ptr(scratch), floats)
    return PrefillLaunch(out, args, keep=(q, cache_k, cache_v, packed, page_table, plan_dev, flags, scratch))


class PrefillLaunch:
    """One validated prefill launch (plan uploaded, output and flags
    allocated); ``run()`` enqueues it on the current stream and returns the
    output.  Repeated runs reuse the same buffers."""

    def __init__(self, out, args, keep=()):
        self.out, self._args, self._keep = out, args, keep
        self._index = out.get_device()

    def run(self):
        return self.phase(3)

    def phase(self, which):
        """Enqueue one phase of the call: 1 the attention kernel (and the merge
        of split items), 2 the exact re-run of flagged items that it did not
        recompute itself (both together = run())."""
        if self._args is not None:
            call('dd_prefill_attention_split', *self._args, int(which), _native.stream_on(self._index))
        return self.out


_CU_COUNT = {}


def _persistent_workgroups(device, dim):
    """Workgroup count for a persistent prefill schedule: one per CU for the
    kernel that runs its items in turn (head sizes up to 128, and 256), else 0."""
    if dim > 256:
        return 0
    forced = os.environ.get('DAMENDAEMON_AMD_PREFILL_WORKGROUPS')   # tuning: 0 = one item per workgroup
    if forced is not None:
        return int(forced)
    return _cu_count(device)


def _cu_count(device):
    index = torch.device(device).index
    index = torch.cuda.current_device() if index is None else index
    if index not in _CU_COUNT:
        _CU_COUNT[index] = torch.cuda.get_device_properties(index).multi_processor_count
    return _CU_COUNT[index]


def prefill_flag_count(segments, max_len, heads, kv_heads, dim, dtype):
    """Entries of the re-run flag workspace a prefill call needs (0: none)."""
    lib = _native.library()
    n = lib.dd_prefill_flag_count(segments, max_len, heads, kv_heads, dim, DTYPE_CODES[dtype])
    if n < 0:
        raise _native.NativeError(f'dd_prefill_flag_count failed: {lib.dd_error_string(-n).decode()} ({-n})')
    return n


def ragged_attention(query, cache_k, cache_v, packed, page_table, window=0, scale=None):
    """Mixed batch: the trailing single-token segments decode, the rest prefill.

    Returns (T, H, D) in the query dtype.  The prefill chunks run before the
    decode rows on the caller's stream.  (Side by side on two streams they gain
    nothing: a prefill workgroup fills a CU's LDS and registers, so a decode
    workgroup only gets onto CUs that have none, and the events between the
    streams cost the host more than the tails that overlap.  8 chunks of 512
    tokens and 120 rows, with pack and rope: 571-588 us on two streams,
    548-552 on one.)
    """
    q = _check(query, cache_k, cache_v, page_table)
    T, H, D = q.shape
    out = torch.empty_like(q)
    lengths = packed.lengths
    n = len(lengths)
    first_decode = n
    while first_decode > 0 and lengths[first_decode - 1] == 1:
        first_decode -= 1
    if first_decode > 0:
        _prepare_prefill(q, cache_k, cache_v, packed, page_table, window, scale, out, (0, first_decode), None).run()
    if first_decode < n:
        rows = slice(sum(lengths[:first_decode]), T)
        kernels.prepare_attention(q[rows].unsqueeze(2), cache_k, cache_v, packed.positions[rows],
                                  packed.slot_ids[rows], window=window, scale=scale, page_table=page_table,
                                  out=out[rows].unsqueeze(2)).run()
    return out
