// Shared pieces of the chunked-prefill kernels (prefill.hip,
// prefill_pipe.hip): the launch parameters, the plan entry of a work item,
// 16-bit output packing and buffer-resource constants.
#pragma once

#include "prefill_f32_item.h"

// The running max of a column is only moved when a tile's max exceeds it by
// more than 2^kMaxSlack in the exp2 domain: probabilities then stay <= 2^8
// (exact in fp32 sums and bf16/f16 operands), and O and l are rescaled a few
// times per column instead of on almost every tile.
constexpr float kMaxSlack = 8.f;

namespace dd_prefill {


constexpr float kNegInf = -__builtin_inff();

struct PrefillParams {
  const void *q;       // (T, H, D)
  const void *k;       // (capacity, KH, page, D)
  const void *v;
  const int64_t *cu;   // (n+1) cu_seqlens of the packed tokens
  const int64_t *ctx;  // (n) start + len
  const int64_t *slots;
  const int32_t *table;
  const int32_t *plan;  // optional: kPlanInts ints per workgroup (see PrefillItem), item -1 = none
  void *out;           // (T, H, D)
  long capacity;
  int n, max_tiles;
  int H, KH, G;
  int page, page_shift;
  int table_w, table_rows;
  int window;
  float scale_log2;     // |scale| * log2(e)
  unsigned q_sign;      // 0x80008000 when scale < 0: q enters negated (exact), so logits use |scale|
  int32_t *flags;       // bf16 pages, D 64/128: per work item, 1 = result must be recomputed exactly
  // Without a plan, a work item's key tiles may be split over max_splits
  // workgroups of split_tiles tiles each (max_splits 1: not split), whose
  // partial results go to `part` and are combined by prefill_merge_kernel.
  int split_tiles, max_splits;
  float *part;
};

// One work item of the prefill kernels: query tile qt of group grp =
// (segment seg, KV head).  A plan entry (dd_prefill_plan) carries the item
// and its segment's token offset, length, start and slot, so that a
// workgroup reads them with one load instead of a chain of two.
constexpr int kPlanInts = DD_PREFILL_PLAN_INTS;   // item, tok0, len, start, slot, rounds, 2 unused
struct PrefillItem {
  int grp, qt, seg, len, start, split;
  long tok0, slot;
};
DD_DEV void prefill_segment(const PrefillParams &p, PrefillItem &it) {
  it.seg = it.grp / p.KH;
  it.tok0 = p.cu[it.seg];
  it.len = (int)(p.cu[it.seg + 1] - it.tok0);
  it.start = (int)p.ctx[it.seg] - it.len;
  it.slot = p.slots[it.seg];
}
// Work items per workgroup under a plan: the plan holds `rounds` entries per
// workgroup, round-major (entry round * gridDim.x + blockIdx.x); every entry
// stores the count (field 5).
DD_DEV int prefill_rounds(const PrefillParams &p) { return p.plan[(long)kPlanInts * blockIdx.x + 5]; }
// Item of round `round` of this workgroup; false: nothing to do.  Without a
// plan workgroup b is unit (split, query tile, group), groups innermost:
// consecutive workgroups go to the 8 XCDs round-robin, each with its own L2,
// so with KV heads in multiples of 8 all units that read one KV head's keys
// share an L2, and every XCD gets the same share of the long segments, of the
// late query tiles and of the first (full) splits, which start first.  (Runs
// of consecutive units per XCD kept the L2 as well, but gave an XCD one
// segment's heads: 8 ragged fp32 segments left CUs idle 36 % of the time.)
template <bool PLAN>
DD_DEV bool prefill_item(const PrefillParams &p, PrefillItem &it, int round) {
  if constexpr (PLAN) {
    const int32_t *e = p.plan + (long)kPlanInts * ((long)round * gridDim.x + blockIdx.x);
    const int item = e[0];
    if (item < 0) return false;
    it.grp = item / p.max_tiles;
    it.qt = item - it.grp * p.max_tiles;
    it.seg = it.grp / p.KH;
    it.tok0 = e[1];
    it.len = e[2];
    it.start = e[3];
    it.slot = e[4];
    it.split = 0;
    return it.grp < p.n * p.KH;
  } else {
    const int ngrp = p.n * p.KH;
    const int r = blockIdx.x / ngrp;
    it.grp = blockIdx.x - r * ngrp;
    it.split = r / p.max_tiles;
    it.qt = p.max_tiles - 1 - (r - it.split * p.max_tiles);
    prefill_segment(p, it);
    return true;
  }
}

// Key tiles kt_first .. kt_last of a work item of query rows r0 .. + rows_here,
// narrowed to its split's share; the number of splits the item has (its last
// split, should the caller's max_splits be too small for it, takes the rest).
template <bool SPLIT>
DD_DEV int prefill_tiles(const PrefillParams &p, const PrefillItem &it, int kt, int r0, int rows_here, int &kt_first,
                         int &kt_last) {
  const int k_hi = it.start + r0 + rows_here;  // exclusive
  const int k_lo = p.window > 0 ? max(0, it.start + r0 - p.window + 1) : 0;
  kt_first = k_lo / kt;
  kt_last = (k_hi - 1) / kt;
  if (!SPLIT) return 1;
  const int nsplit = min((kt_last - kt_first) / p.split_tiles + 1, p.max_splits);
  kt_first += it.split * p.split_tiles;
  if (it.split + 1 < nsplit) kt_last = kt_first + p.split_tiles - 1;
  return nsplit;
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

template <int DT>
DD_DEV unsigned pack2(float a, float b) {
  if constexpr (DT == DD_BF16) {
    return (unsigned)float_to_bf16_bits(a) | ((unsigned)float_to_bf16_bits(b) << 16);
  } else {
    return (unsigned)float_to_f16_bits(a) | ((unsigned)float_to_f16_bits(b) << 16);
  }
}

// A flagged item again, in fp32 arithmetic and in place (LDS: f32_lds<D>()
// bytes free for it).  The whole workgroup of W = 8 waves calls it; up to 128
// query heads per KV head (prefill_redo_fits), beyond that the flags are left
// to prefill_f32_kernel's launch, which costs 4 us of every call to look for
// them.  (The code beside the hot loop costs the planned kernel about 1 %: 8 x
// 512 tokens 226.8 us in one launch, 224.8 + 4 in two.)
constexpr bool prefill_redo_fits(int G) { return G <= 128; }
template <int DT, int D, int W>
DD_DEV void prefill_redo(const PrefillParams &p, char *lds, int grp, int r0, int end) {
  PrefillGenericArgs a{};
  a.q = p.q;
  a.k = p.k;
  a.v = p.v;
  a.cu = p.cu;
  a.ctx = p.ctx;
  a.slots = p.slots;
  a.table = p.table;
  a.out = p.out;
  a.capacity = p.capacity;
  a.n = p.n;
  a.heads = p.H;
  a.kv_heads = p.KH;
  a.dim = D;
  a.page = p.page;
  a.page_shift = p.page_shift;
  a.table_w = p.table_w;
  a.table_rows = p.table_rows;
  a.window = p.window;
  a.scale_log2 = p.q_sign ? -p.scale_log2 : p.scale_log2;
  for (int r = r0; r < end; r += 16 * W / p.G) {
    __syncthreads();   // the previous users' LDS reads are done
    f32_item<DT, D, W>(a, lds, grp, r, end);
  }
}

// Floats of one split's partial result: per wave of `columns` / 32, 32 columns
// of O^T over whole 32-dim blocks, in accumulator order ((dim block, register
// quad), lane), then the 32 running offsets and the 32 denominators.
constexpr long prefill_part_floats(int columns, int dim) {
  return (long)(columns / 32) * (32L * ((dim + 31) / 32 * 32) + 64);
}

// 32-bit word 3 of a raw (untyped) buffer resource.
constexpr int kBufferWord3 = 0x00020000;

typedef __attribute__((address_space(3))) void lds_void;

// Keys per tile of prefill_x3_kernel (its columns per work item: 256).
#define DD_PREFILL_X3_KEYS 32
// Below this a whole result row may miss the parts of V under 2^-126 that its
// bf16 products lose (2^-26 of it).
constexpr float kX3Least = 0x1p-100f;

int prefill_pipe_dispatch(const PrefillParams &p, int dtype, int dim, int max_len, int plan_len, hipStream_t s);
int prefill_x3_dispatch(const PrefillParams &p, int dim, int max_len, hipStream_t s);

}  // namespace dd_prefill
