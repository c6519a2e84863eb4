// The combine of split prefill work items (prefill_pipe.hip, prefill_x3.hip).
#pragma once

#include "prefill_common.h"

namespace dd_prefill {
namespace {

// Combines the splits of the work items that have several: workgroup (item,
// w) holds the 32 columns of wave w of the split kernel, its wave md their
// dims 32 md ..+32, each lane the four-dim pieces it held there, so every
// load is 1 KiB of consecutive bytes.  Reads kBatch splits at a time (all
// loads in flight), as the decode merge does.  Items whose result has to be
// recomputed exactly raise their flag: bf16 ones that show V outside fp16's
// normal range (see prefill_pipe_kernel), fp32 ones that are not finite or tiny
// (see prefill_x3_kernel).  NW, KT: waves and keys per tile of the split kernel.
template <int DT, int NW, int KT, int DR>
__global__ __launch_bounds__(64 * ((DR + 31) / 32)) void prefill_merge_kernel(PrefillParams p) {
  constexpr int MDR = (DR + 31) / 32;
  constexpr int COLS = 32 * NW;
  constexpr int kBatch = 4;
  __shared__ unsigned s_top[MDR][32];
  const int lane = threadIdx.x & 63;
  const int md = uniform(threadIdx.x >> 6);
  const int l32 = lane & 31, h2 = lane >> 5;
  const int w = blockIdx.y;
  PrefillItem it;
  it.grp = blockIdx.x / p.max_tiles;
  it.qt = blockIdx.x - it.grp * p.max_tiles;
  it.split = 0;
  prefill_segment(p, it);
  const int G = p.G;
  const int rows = COLS / G;
  const int r0 = it.qt * rows;
  if (r0 >= it.len) return;
  const int rows_here = min(rows, it.len - r0);
  int kt_first, kt_last;
  const int nsplit = prefill_tiles<true>(p, it, KT, r0, rows_here, kt_first, kt_last);
  if (nsplit <= 1 || 32 * w / G >= rows_here) return;
  const int col = w * 32 + l32;
  const int qr = col / G, gh = col - (col / G) * G;
  const bool colok = qr < rows_here;

  const long step = prefill_part_floats(COLS, DR);
  const float *part = p.part + (long)blockIdx.x * p.max_splits * step + (long)w * prefill_part_floats(32, DR);
  float m = kNegInf, l = 0.f;
  f32x4 o[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) o[q] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < nsplit; s0 += kBatch) {
    float ms[kBatch], ls[kBatch];
    f32x4 os[kBatch][4];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const float *src = part + min(s0 + j, nsplit - 1) * step;   // (clamped; weight 0 below)
      ms[j] = src[1024 * MDR + l32];
      ls[j] = src[1024 * MDR + 32 + l32];
#pragma unroll
      for (int q = 0; q < 4; ++q) os[j][q] = ((const f32x4 *)src)[(md * 4 + q) * 64 + lane];
    }
    float top = m;
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      if (s0 + j >= nsplit) ms[j] = kNegInf;
      top = fmaxf(top, ms[j]);
    }
    const float base = top == kNegInf ? 0.f : top;
    const float a = __builtin_amdgcn_exp2f(m - base);
    l *= a;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] *= a;
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      if (s0 + j >= nsplit) break;
      const float x = __builtin_amdgcn_exp2f(ms[j] - base);   // 0 where the split had no key for the column
      l += x * ls[j];
#pragma unroll
      for (int q = 0; q < 4; ++q) o[q] += x * os[j][q];
    }
    m = top;
  }
  if constexpr (DT != DD_F16) {
    if (p.flags) {
      unsigned mb = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) mb = max(mb, __float_as_uint(o[q][i]) & 0x7fffffffu);
      mb = max(mb, (unsigned)__shfl_xor((int)mb, 32));
      if (h2 == 0) s_top[md][l32] = mb;
      __syncthreads();
      if (md == 0) {
#pragma unroll
        for (int k = 1; k < MDR; ++k) mb = max(mb, s_top[k][l32]);
        const float top = __uint_as_float(mb) / l;
        const bool fine = top >= (DT == DD_F32 ? kX3Least : 0x1p-12f) && top <= 3.0e38f;
        if (__builtin_amdgcn_ballot_w64(colok && !fine) && lane == 0)
          p.flags[blockIdx.x] = 1;
      }
    }
  }
  if (!colok) return;
  const float inv = 1.f / l;
  const long row = ((it.tok0 + r0 + qr) * p.H + (long)(it.grp - it.seg * p.KH) * G + gh) * DR;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int d = 32 * md + 8 * q + 4 * h2;
    if (DR % 32 && d >= DR) continue;
    if constexpr (DT == DD_F32)
      *(f32x4 *)((float *)p.out + row + d) = o[q] * inv;
    else
      *(u32x2 *)((unsigned short *)p.out + row + d) =
          u32x2{pack2<DT>(o[q][0] * inv, o[q][1] * inv), pack2<DT>(o[q][2] * inv, o[q][3] * inv)};
  }
}

}  // namespace
}  // namespace dd_prefill
