// Ragged-batch packer and K/V page writer for gfx950.
//
// The packer replaces the host-side list comprehensions of
// damendaemon/paged.py:149-159 (and batch.py:133-136), the segment ends of
// paged.py:118-120 and the in-kernel slot computation of kernels.py:279-281.
// For n segments (slot_i, start_i, len_i) it writes, bit-exactly:
//   cu_seqlens[i]  = len_0 + ... + len_{i-1}          (n+1 entries)
//   ends[i]        = cu_seqlens[i+1] - 1
//   context[i]     = start_i + len_i
//   positions[t]   = start_i + (t - cu_seqlens[i])    for t in segment i
//   slot_ids[t]    = slot_i
//   slot_map[t]    = table[slot_i, pos / P] * P + pos % P
//   cu_pages[i]    = sum_{j<i} ceil(context_j / P)    (n+1 entries)
//   gather[k]      = table[slot_i, k - cu_pages[i]]   (physical pages of each
//                    segment's whole history, in logical order)
// Segment-level prefix sums run in one workgroup (wave-level scans through
// LDS); the per-token and per-page outputs are filled by a grid of
// workgroups that locate their segment by binary search in the prefix.
//
// Segments known on the host (dd_pack_batch_host) travel in the kernel's own
// arguments, kPackSegs per launch, and one launch fills everything: every
// workgroup scans the launch's segments in LDS (no segment waits for another
// launch's scan), so there is no upload and no second launch.
#include "common.h"
#include "q8.h"

namespace {

constexpr int kScanThreads = 1024;

// Inclusive scan of one int64 per thread across the workgroup.
DD_DEV long block_scan(long x, long *s_tmp) {
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const long y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) s_tmp[w] = x;
  __syncthreads();
  if (w == 0) {
    long t = lane < (int)(blockDim.x >> 6) ? s_tmp[lane] : 0;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const long y = __shfl_up(t, off, 64);
      if (lane >= off) t += y;
    }
    if (lane < (int)(blockDim.x >> 6)) s_tmp[lane] = t;
  }
  __syncthreads();
  if (w > 0) x += s_tmp[w - 1];
  __syncthreads();
  return x;
}

__global__ __launch_bounds__(kScanThreads) void scan_kernel(const int64_t *lengths, const int64_t *starts, int n,
                                                            int page, int64_t *cu, int64_t *ends,
                                                            int64_t *context, int32_t *cu_pages) {
  __shared__ long s_tmp[16];
  __shared__ long s_carry[2];
  if (threadIdx.x == 0) {
    s_carry[0] = 0;
    s_carry[1] = 0;
    cu[0] = 0;
    if (cu_pages) cu_pages[0] = 0;
  }
  __syncthreads();
  for (int base = 0; base < n; base += kScanThreads) {
    const int i = base + threadIdx.x;
    const long len = i < n ? lengths[i] : 0;
    const long ctx = i < n ? starts[i] + len : 0;
    const long np = (ctx + page - 1) / page;
    const long c0 = s_carry[0], c1 = s_carry[1];
    __syncthreads();
    const long inc_t = block_scan(len, s_tmp) + c0;
    const long inc_p = block_scan(i < n ? np : 0, s_tmp) + c1;
    if (i < n) {
      cu[i + 1] = inc_t;
      ends[i] = inc_t - 1;
      context[i] = ctx;
      if (cu_pages) cu_pages[i + 1] = (int32_t)inc_p;
    }
    if (threadIdx.x == kScanThreads - 1) {
      s_carry[0] = inc_t;
      s_carry[1] = inc_p;
    }
    __syncthreads();
  }
}

// Index of the segment whose [cu[i], cu[i+1]) holds t (cu ascending).
template <typename T>
DD_DEV int find_segment(const T *cu, int n, long t) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((long)cu[mid] <= t) lo = mid; else hi = mid - 1;
  }
  return lo;
}

__global__ __launch_bounds__(256) void fill_tokens_kernel(const int64_t *cu, const int64_t *starts,
                                                          const int64_t *slots, int n, long total,
                                                          const int32_t *table, int table_rows, int table_w,
                                                          int page, int64_t *positions, int64_t *slot_ids,
                                                          int64_t *slot_map) {
  const long t = (long)blockIdx.x * 256 + threadIdx.x;
  if (t >= total) return;
  int i = find_segment(cu, n, t);
  // empty segments share their cu value with the next one: skip forward
  while (i + 1 < n && cu[i + 1] <= t) ++i;
  const long pos = starts[i] + (t - cu[i]);
  const long slot = slots[i];
  positions[t] = pos;
  slot_ids[t] = slot;
  if (slot_map) {
    const long entry = pos / page;
    long phys = -1;
    if (slot >= 0 && slot < table_rows && entry < table_w) phys = table[slot * table_w + entry];
    slot_map[t] = phys * page + pos % page;
  }
}

__global__ __launch_bounds__(256) void fill_pages_kernel(const int32_t *cu_pages, const int64_t *slots, int n,
                                                         long total, const int32_t *table, int table_rows,
                                                         int table_w, int32_t *gather) {
  const long k = (long)blockIdx.x * 256 + threadIdx.x;
  if (k >= total) return;
  int i = find_segment(cu_pages, n, k);
  while (i + 1 < n && cu_pages[i + 1] <= k) ++i;
  const long slot = slots[i];
  const long entry = k - cu_pages[i];
  gather[k] = (slot >= 0 && slot < table_rows && entry < table_w) ? table[slot * table_w + entry] : -1;
}

// Segments of one dd_pack_batch_host launch: numbers i0 .. i0 + n of the batch,
// the first of them at token tok0 and gather entry page0.
constexpr int kPackSegs = 256;
struct PackSegs {
  int n, i0, total;      // total: segments of the whole batch (row stride of meta)
  int tok_blocks;        // workgroups of the tokens; the ones after them fill the page gather
  long tok0, page0;
  int len[kPackSegs], start[kPackSegs], slot[kPackSegs];
};
struct PackOut {
  int64_t *cu, *ends, *context, *meta, *positions, *slot_ids, *slot_map;
  int32_t *cu_pages, *gather;
};

__global__ __launch_bounds__(kPackSegs) void pack_segments_kernel(PackSegs segs, const int32_t *table, int table_rows,
                                                                  int table_w, int page, PackOut out) {
  __shared__ long s_tmp[16];
  __shared__ int s_cu[kPackSegs + 1], s_cp[kPackSegs + 1], s_start[kPackSegs], s_slot[kPackSegs];
  const int i = threadIdx.x;
  const int len = i < segs.n ? segs.len[i] : 0;
  const int start = i < segs.n ? segs.start[i] : 0;
  const int slot = i < segs.n ? segs.slot[i] : 0;
  const long ctx = (long)start + len;
  const int np = (int)((ctx + page - 1) / page);
  // both prefix sums in one scan: tokens in the low half, pages in the high one
  const long both = block_scan((long)len | ((long)np << 32), s_tmp);
  const int cu = (int)both, cp = (int)(both >> 32);
  s_cu[i + 1] = cu;
  s_cp[i + 1] = cp;
  s_start[i] = start;
  s_slot[i] = slot;
  if (i == 0) s_cu[0] = s_cp[0] = 0;
  __syncthreads();
  if (blockIdx.x == 0 && i < segs.n) {
    const int g = segs.i0 + i;
    out.cu[g + 1] = segs.tok0 + cu;
    out.ends[g] = segs.tok0 + cu - 1;
    out.context[g] = ctx;
    out.meta[g] = len;
    out.meta[segs.total + g] = start;
    out.meta[2L * segs.total + g] = slot;
    if (out.cu_pages) out.cu_pages[g + 1] = (int32_t)(segs.page0 + cp);
    if (g == 0) {
      out.cu[0] = 0;
      if (out.cu_pages) out.cu_pages[0] = 0;
    }
  }
  if ((int)blockIdx.x < segs.tok_blocks) {
    const int t = blockIdx.x * kPackSegs + i;
    if (t >= s_cu[segs.n]) return;
    int k = find_segment(s_cu, segs.n, t);
    while (k + 1 < segs.n && s_cu[k + 1] <= t) ++k;   // (empty segments)
    const long pos = (long)s_start[k] + (t - s_cu[k]);
    const long sl = s_slot[k];
    out.positions[segs.tok0 + t] = pos;
    out.slot_ids[segs.tok0 + t] = sl;
    if (out.slot_map) {
      const long entry = pos / page;
      long phys = -1;
      if (sl >= 0 && sl < table_rows && entry < table_w) phys = table[sl * table_w + entry];
      out.slot_map[segs.tok0 + t] = phys * page + (pos - entry * page);
    }
    return;
  }
  const int e = ((int)blockIdx.x - segs.tok_blocks) * kPackSegs + i;
  if (e >= s_cp[segs.n]) return;
  int k = find_segment(s_cp, segs.n, e);
  while (k + 1 < segs.n && s_cp[k + 1] <= e) ++k;
  const long sl = s_slot[k];
  const long entry = e - s_cp[k];
  out.gather[segs.page0 + e] = (sl >= 0 && sl < table_rows && entry < table_w) ? table[sl * table_w + entry] : -1;
}

// One thread moves 16 bytes of one (token, KV head) row into its page slot.
__global__ __launch_bounds__(256) void store_pages_kernel(const char *key, const char *value,
                                                          const int64_t *slot_map, long tokens, int kv_heads,
                                                          int row_bytes, int page, long capacity, char *ck,
                                                          char *cv) {
  const int per_row = row_bytes / 16;
  const long g = (long)blockIdx.x * 256 + threadIdx.x;
  const long per_token = (long)kv_heads * per_row;
  if (g >= tokens * per_token) return;
  const long t = g / per_token;
  const int rem = (int)(g - t * per_token);
  const int kh = rem / per_row;
  const int chunk = rem - kh * per_row;
  const long s = slot_map[t];
  if (s < 0) return;
  const long phys = s / page;
  if (phys >= capacity) return;
  const long dst = ((phys * kv_heads + kh) * page + (s % page)) * (long)row_bytes + 16L * chunk;
  const long src = (t * kv_heads + kh) * (long)row_bytes + 16L * chunk;
  *(u32x4 *)(ck + dst) = *(const u32x4 *)(key + src);
  *(u32x4 *)(cv + dst) = *(const u32x4 *)(value + src);
}

// One thread quantises one (token, KV head, channel group) of K and of V
// straight into int8 pages and their fp16 scale rows.
template <int DT>
__global__ __launch_bounds__(256) void store_pages_q8_kernel(const void *key, const void *value,
                                                             const int64_t *slot_map, long tokens, int kv_heads,
                                                             int dim, int group, int page, long capacity,
                                                             signed char *ck, signed char *cv,
                                                             unsigned short *ks, unsigned short *vs) {
  const int ng = dim / group;
  const long g = (long)blockIdx.x * 256 + threadIdx.x;
  const long per_token = (long)kv_heads * ng;
  if (g >= tokens * per_token) return;
  const long t = g / per_token;
  const int rem = (int)(g - t * per_token);
  const int kh = rem / ng;
  const int gi = rem - kh * ng;
  const long s = slot_map[t];
  if (s < 0 || s / page >= capacity) return;
  const long row = ((s / page) * kv_heads + kh) * page + (s % page);
  const long src = (t * kv_heads + kh) * (long)dim + (long)gi * group;
  const long dst = row * dim + (long)gi * group;
  ks[row * ng + gi] = q8_group<DT>(key, src, group, ck + dst);
  vs[row * ng + gi] = q8_group<DT>(value, src, group, cv + dst);
}

// The same with eight channels per lane and 2^shift lanes per group (q8.h):
// lane i of n = (tokens * kv_heads * groups) << shift.
template <int DT>
__global__ __launch_bounds__(256) void store_pages_q8_lanes_kernel(const void *key, const void *value,
                                                                   const int64_t *slot_map, unsigned n,
                                                                   unsigned per_token, int kv_heads, int dim,
                                                                   int group, int shift, int page, long capacity,
                                                                   signed char *ck, signed char *cv,
                                                                   unsigned short *ks, unsigned short *vs) {
  const unsigned i = blockIdx.x * 256u + threadIdx.x;
  const unsigned g = i >> shift;
  const int c = 8 * (int)(i & ((1u << shift) - 1));
  const unsigned ng = (unsigned)(dim / group);
  const unsigned t = g / per_token, rem = g - t * per_token;
  const unsigned kh = rem / ng, gi = rem - kh * ng;
  const bool in = i < n && c < group;
  const long s = in ? slot_map[t] : -1;
  const long phys = s < 0 ? -1 : s <= 0x7fffffffL ? (long)((unsigned)s / (unsigned)page) : s / page;
  const bool on = s >= 0 && phys < capacity;
  const long src = (long)g * group + c;      // (token, KV head, group) rows are contiguous
  float k[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (in) {
    q8_load8<DT>(key, src, k);
    q8_load8<DT>(value, src, v);
  }
  unsigned short kbits, vbits;
  const u32x2 kq = q8_lanes(k, shift, &kbits), vq = q8_lanes(v, shift, &vbits);
  if (!on) return;
  const long row = (phys * kv_heads + kh) * page + (s - phys * page);
  *(u32x2 *)(ck + row * dim + gi * group + c) = kq;
  *(u32x2 *)(cv + row * dim + gi * group + c) = vq;
  if (c == 0) {
    ks[row * ng + gi] = kbits;
    vs[row * ng + gi] = vbits;
  }
}

}  // namespace

extern "C" int dd_pack_batch(const int64_t *lengths, const int64_t *starts, const int64_t *slots, int n,
                             int64_t total_tokens, int64_t total_pages, const int32_t *page_table,
                             int table_rows, int table_width, int page_size, int64_t *cu_seqlens, int64_t *ends,
                             int64_t *context_lens, int64_t *positions, int64_t *slot_ids, int64_t *slot_map,
                             int32_t *cu_pages, int32_t *gather_pages, void *stream) {
  if (n < 0 || total_tokens < 0 || page_size <= 0 || !cu_seqlens) return DD_EINVAL;
  if (n > 0 && (!lengths || !starts || !slots || !ends || !context_lens)) return DD_EINVAL;
  if ((slot_map || gather_pages) && (!page_table || table_width <= 0)) return DD_EINVAL;
  if (gather_pages && !cu_pages) return DD_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(scan_kernel, dim3(1), dim3(kScanThreads), 0, s, lengths, starts, n, page_size, cu_seqlens,
                     ends, context_lens, cu_pages);
  DD_LAUNCH_CHECK();
  if (n > 0 && total_tokens > 0) {
    if (!positions || !slot_ids) return DD_EINVAL;
    hipLaunchKernelGGL(fill_tokens_kernel, dim3((unsigned)dd_cdiv(total_tokens, 256)), dim3(256), 0, s,
                       cu_seqlens, starts, slots, n, (long)total_tokens, page_table, table_rows, table_width,
                       page_size, positions, slot_ids, slot_map);
    DD_LAUNCH_CHECK();
  }
  if (n > 0 && gather_pages && total_pages > 0) {
    hipLaunchKernelGGL(fill_pages_kernel, dim3((unsigned)dd_cdiv(total_pages, 256)), dim3(256), 0, s, cu_pages,
                       slots, n, (long)total_pages, page_table, table_rows, table_width, gather_pages);
    DD_LAUNCH_CHECK();
  }
  return DD_OK;
}

extern "C" int dd_pack_batch_host(const int64_t *lengths, const int64_t *starts, const int64_t *slots, int n,
                                  int64_t total_tokens, int64_t total_pages, const int32_t *page_table,
                                  int table_rows, int table_width, int page_size, int64_t *cu_seqlens, int64_t *ends,
                                  int64_t *context_lens, int64_t *meta, int64_t *positions, int64_t *slot_ids,
                                  int64_t *slot_map, int32_t *cu_pages, int32_t *gather_pages, void *stream) {
  if (n <= 0 || !lengths || !starts || !slots || page_size <= 0 || !cu_seqlens || !ends || !context_lens || !meta)
    return DD_EINVAL;
  if ((slot_map || gather_pages) && (!page_table || table_width <= 0)) return DD_EINVAL;
  if (gather_pages && !cu_pages) return DD_EINVAL;
  // 32-bit segments whose sums fit (anything larger: dd_pack_batch), and totals
  // that are theirs
  constexpr int64_t kMax = 0x3fffffff;
  int64_t tokens = 0, pages = 0;
  for (int i = 0; i < n; ++i) {
    if (lengths[i] < 0 || starts[i] < 0) return DD_EINVAL;
    if (lengths[i] > kMax || starts[i] > kMax || slots[i] < -kMax || slots[i] > kMax) return DD_EUNSUPPORTED;
    tokens += lengths[i];
    pages += (lengths[i] + starts[i] + page_size - 1) / page_size;
    if (tokens > kMax || pages > kMax) return DD_EUNSUPPORTED;
  }
  if (tokens != total_tokens || (gather_pages && pages != total_pages)) return DD_EINVAL;
  if (tokens > 0 && (!positions || !slot_ids)) return DD_EINVAL;
  const PackOut out{cu_seqlens, ends, context_lens, meta, positions, slot_ids, slot_map, cu_pages, gather_pages};
  PackSegs segs;
  segs.total = n;
  segs.tok0 = segs.page0 = 0;
  for (segs.i0 = 0; segs.i0 < n; segs.i0 += kPackSegs) {
    segs.n = n - segs.i0 < kPackSegs ? n - segs.i0 : kPackSegs;
    int64_t t = 0, pg = 0;
    for (int i = 0; i < segs.n; ++i) {
      const int64_t len = lengths[segs.i0 + i], start = starts[segs.i0 + i];
      segs.len[i] = (int)len;
      segs.start[i] = (int)start;
      segs.slot[i] = (int)slots[segs.i0 + i];
      t += len;
      pg += (len + start + page_size - 1) / page_size;
    }
    segs.tok_blocks = (int)dd_cdiv(t, kPackSegs);
    const long grid = segs.tok_blocks + (gather_pages ? dd_cdiv(pg, kPackSegs) : 0);
    hipLaunchKernelGGL(pack_segments_kernel, dim3((unsigned)(grid > 0 ? grid : 1)), dim3(kPackSegs), 0,
                       (hipStream_t)stream, segs, page_table, table_rows, table_width, page_size, out);
    DD_LAUNCH_CHECK();
    segs.tok0 += t;
    segs.page0 += pg;
  }
  return DD_OK;
}

extern "C" int dd_store_kv_pages(const void *key, const void *value, int elem_bytes, const int64_t *slot_map,
                                 int64_t tokens, int kv_heads, int dim, int page_size, int64_t capacity,
                                 void *cache_k, void *cache_v, void *stream) {
  if (!key || !value || !slot_map || !cache_k || !cache_v || tokens < 0 || kv_heads <= 0 || dim <= 0 ||
      page_size <= 0 || capacity <= 0 || (elem_bytes != 1 && elem_bytes != 2 && elem_bytes != 4))
    return DD_EINVAL;
  const int row_bytes = dim * elem_bytes;
  if (row_bytes % 16) return DD_EUNSUPPORTED;
  const long work = (long)tokens * kv_heads * (row_bytes / 16);
  if (work == 0) return DD_OK;
  hipLaunchKernelGGL(store_pages_kernel, dim3((unsigned)dd_cdiv(work, 256)), dim3(256), 0, (hipStream_t)stream,
                     (const char *)key, (const char *)value, slot_map, (long)tokens, kv_heads, row_bytes,
                     page_size, (long)capacity, (char *)cache_k, (char *)cache_v);
  DD_LAUNCH_CHECK();
  return DD_OK;
}

extern "C" int dd_store_kv_pages_q8(const void *key, const void *value, int dtype, const int64_t *slot_map,
                                    int64_t tokens, int kv_heads, int dim, int group, int page_size,
                                    int64_t capacity, void *cache_k, void *cache_v, void *k_scale, void *v_scale,
                                    void *stream) {
  if (!key || !value || !slot_map || !cache_k || !cache_v || !k_scale || !v_scale || tokens < 0 ||
      kv_heads <= 0 || dim <= 0 || group <= 0 || dim % group || page_size <= 0 || capacity <= 0)
    return DD_EINVAL;
  const long work = (long)tokens * kv_heads * (dim / group);
  if (work == 0) return DD_OK;
  hipStream_t s = (hipStream_t)stream;
  auto *ck = (signed char *)cache_k;
  auto *cv = (signed char *)cache_v;
  auto *ks = (unsigned short *)k_scale;
  auto *vs = (unsigned short *)v_scale;
  // eight channels per lane where rows start on 16 bytes and the lanes fit 32 bits
  const int shift = q8_lane_shift(group);
  if (shift >= 0 && (work << shift) <= 0x7fffffffL && dd_aligned(key, 16) && dd_aligned(value, 16) &&
      dd_aligned(cache_k, 8) && dd_aligned(cache_v, 8)) {
    const unsigned n = (unsigned)(work << shift);
    const dim3 lanes((unsigned)dd_cdiv(n, 256));
#define DD_Q8_LANES(DT)                                                                                          \
  hipLaunchKernelGGL(store_pages_q8_lanes_kernel<DT>, lanes, dim3(256), 0, s, key, value, slot_map, n,           \
                     (unsigned)(kv_heads * (dim / group)), kv_heads, dim, group, shift, page_size, (long)capacity, \
                     ck, cv, ks, vs)
    switch (dtype) {
      case DD_F32: DD_Q8_LANES(DD_F32); break;
      case DD_F16: DD_Q8_LANES(DD_F16); break;
      case DD_BF16: DD_Q8_LANES(DD_BF16); break;
      default: return DD_EUNSUPPORTED;
    }
#undef DD_Q8_LANES
    DD_LAUNCH_CHECK();
    return DD_OK;
  }
  const dim3 grid((unsigned)dd_cdiv(work, 256));
#define DD_Q8_STORE(DT)                                                                                    \
  hipLaunchKernelGGL(store_pages_q8_kernel<DT>, grid, dim3(256), 0, s, key, value, slot_map, (long)tokens, \
                     kv_heads, dim, group, page_size, (long)capacity, ck, cv, ks, vs)
  switch (dtype) {
    case DD_F32: DD_Q8_STORE(DD_F32); break;
    case DD_F16: DD_Q8_STORE(DD_F16); break;
    case DD_BF16: DD_Q8_STORE(DD_BF16); break;
    default: return DD_EUNSUPPORTED;
  }
#undef DD_Q8_STORE
  DD_LAUNCH_CHECK();
  return DD_OK;
}
