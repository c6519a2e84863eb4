// One work item of chunked prefill in fp32 arithmetic on the matrix cores: the
// body of prefill_f32_kernel (prefill_f32.hip, which describes it), and what
// the other prefill kernels recompute an item with whose operands do not fit
// their 16-bit ones.
#pragma once

#include "common.h"
#include "prefill_generic.h"

namespace {

constexpr int kKT = 32;            // keys per tile
constexpr int kSub = kKT / 16;     // 16-key MFMA tiles per key tile
constexpr float kF32NegInf = -__builtin_inff();
constexpr float kSlack = 8.f;      // running-max slack (exp2 domain)

// Four elements of the given dtype at element index idx, widened to fp32.
template <int DT>
DD_DEV f32x4 load4(const void *base, long idx) {
  if constexpr (DT == DD_F32) {
    return *(const f32x4 *)((const float *)base + idx);
  } else {
    const u32x2 w = *(const u32x2 *)((const unsigned short *)base + idx);
    if constexpr (DT == DD_BF16) {
      return f32x4{bf16_lo(w[0]), __uint_as_float(w[0] & 0xffff0000u), bf16_lo(w[1]),
                   __uint_as_float(w[1] & 0xffff0000u)};
    } else {
      return f32x4{half_bits_to_float((unsigned short)(w[0] & 0xffffu)), half_bits_to_float((unsigned short)(w[0] >> 16)),
                   half_bits_to_float((unsigned short)(w[1] & 0xffffu)), half_bits_to_float((unsigned short)(w[1] >> 16))};
    }
  }
}

// LDS of one item: [buffer][K, V], rows padded by 16 bytes.
template <int D>
constexpr int f32_lds() { return 2 * 2 * kKT * (4 * D + 16); }

// One work item: query rows r0 .. min(r0 + 16 W / G, end) of group grp =
// (segment, KV head).
template <int DT, int D, int W>
DD_DEV void f32_item(const PrefillGenericArgs &p, char *lds, int grp, int r0, int end) {
  typedef char Buffers[2][2][kKT * (4 * D + 16)];
  Buffers &s_kv = *(Buffers *)lds;
  constexpr int NT = 64 * W;
  constexpr int COLS = 16 * W;                     // (query row, head) columns per workgroup
  constexpr int RS = 4 * D + 16;                   // LDS row stride (bytes, padded)
  constexpr int TILEB = kKT * RS;                  // one tile of K (or V)
  constexpr int NC = D / 16;                       // 4-dim Q / K pieces per lane
  constexpr int MD = D / 16;                       // O^T row tiles
  constexpr int PPR = D / 4;                       // 4-element pieces per key row
  constexpr int PCS = (kKT * PPR + NT - 1) / NT;   // pieces per thread and plane
  static_assert(D % 16 == 0 && D <= 256, "head size");


  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = uniform(tid >> 6);
  const int n16 = lane & 15;
  const int kg = lane >> 4;

  const int G = p.heads / p.kv_heads;
  const int rows = COLS / G;
  const int seg = grp / p.kv_heads;
  const int kh = grp - seg * p.kv_heads;
  const long tok0 = p.cu[seg];
  const int len = (int)(p.cu[seg + 1] - tok0);
  end = min(end, len);
  if (r0 >= end) return;
  const int context = (int)p.ctx[seg];
  const int start = context - len;
  const long slot = p.slots[seg];
  const int rows_here = min(rows, end - r0);
  const int k_hi = start + r0 + rows_here;  // exclusive
  const int k_lo = p.window > 0 ? max(0, start + r0 - p.window + 1) : 0;
  const int t_first = k_lo / kKT;
  const int t_last = (k_hi - 1) / kKT;

  // ---- this lane's column and its Q^T operand ----
  const int col = w * 16 + n16;
  const int qr = col / G;
  const int gh = col - qr * G;
  const bool colok = qr < rows_here;
  const int qpos = start + r0 + qr;
  const long qrow = ((tok0 + r0 + (colok ? qr : 0)) * p.heads + (long)kh * G + gh) * D;
  f32x4 qa[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) qa[c] = colok ? load4<DT>(p.q, qrow + (D / 4) * kg + 4 * c) : f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- tile staging: thread piece e = tid + NT j is row e / PPR, dims 4 (e % PPR) ..+4 ----
  const bool slot_ok = slot >= 0 && slot < p.table_rows;
  auto fetch = [&](int t, f32x4 (&kr)[PCS], f32x4 (&vr)[PCS]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < PCS; ++j) {
      const int e = tid + NT * j;
      const int key = t * kKT + e / PPR;
      long base = -1;
      if (e < kKT * PPR && slot_ok && key < context) {
        const int entry = key >> p.page_shift;
        const long phys = entry < p.table_w ? p.table[slot * p.table_w + entry] : -1;
        if (phys >= 0 && phys < p.capacity)
          base = (((phys * p.kv_heads + kh) << p.page_shift) + (key & (p.page - 1))) * (long)D + 4 * (e % PPR);
      }
      kr[j] = base >= 0 ? load4<DT>(p.k, base) : f32x4{0.f, 0.f, 0.f, 0.f};
      vr[j] = base >= 0 ? load4<DT>(p.v, base) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto stage = [&](int buf, const f32x4 (&kr)[PCS], const f32x4 (&vr)[PCS]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < PCS; ++j) {
      const int e = tid + NT * j;
      if (e < kKT * PPR) {
        const int off = (e / PPR) * RS + 16 * (e % PPR);
        *(f32x4 *)(s_kv[buf][0] + off) = kr[j];
        *(f32x4 *)(s_kv[buf][1] + off) = vr[j];
      }
    }
  };

  f32x4 o[MD];
#pragma unroll
  for (int md = 0; md < MD; ++md) o[md] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = kF32NegInf;  // running max of this lane's column (scaled, exp2 domain)
  float lsum = 0.f;       // this lane's share of the column's denominator

  auto compute = [&](int buf, int t) __attribute__((always_inline)) {
    const char *sk = s_kv[buf][0];
    const char *sv = s_kv[buf][1];
    float x[kSub][4];
    float mx = kF32NegInf;
#pragma unroll
    for (int h = 0; h < kSub; ++h) {
      const char *krow = sk + (16 * h + n16) * RS + D * kg;   // dims (D/4) kg ..
      f32x4 ka[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) ka[c] = *(const f32x4 *)(krow + 16 * c);
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) s = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[c][q], qa[c][q], s, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = t * kKT + 16 * h + 4 * kg + i;
        const bool live = colok && key <= qpos && (p.window <= 0 || key > qpos - p.window);
        x[h][i] = live ? s[i] * p.scale_log2 : kF32NegInf;
        mx = fmaxf(mx, x[h][i]);
      }
    }
    mx = xor32_max(xor16_max(mx));
    const bool up = mx > m_run + kSlack;
    if (__builtin_amdgcn_ballot_w64(up)) {
      const float mn = up ? mx : m_run;
      const float alpha = up ? (m_run == kF32NegInf ? 0.f : __builtin_amdgcn_exp2f(m_run - mn)) : 1.f;
      m_run = mn;
      lsum *= alpha;
#pragma unroll
      for (int md = 0; md < MD; ++md) o[md] *= alpha;
    }
    const float mu = m_run == kF32NegInf ? 0.f : m_run;
#pragma unroll
    for (int h = 0; h < kSub; ++h) {
      float pr[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pr[i] = __builtin_amdgcn_exp2f(x[h][i] - mu);
        lsum += pr[i];
      }
      // V of key 16h + 4kg + e, dims MD n16 .. +MD (16-, 8- or 4-byte reads)
      float vf[4][MD];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float *vrow = (const float *)(sv + (16 * h + 4 * kg + e) * RS) + MD * n16;
        if constexpr (MD % 4 == 0) {
#pragma unroll
          for (int q = 0; q < MD / 4; ++q) {
            const f32x4 v4 = *(const f32x4 *)(vrow + 4 * q);
#pragma unroll
            for (int u = 0; u < 4; ++u) vf[e][4 * q + u] = v4[u];
          }
        } else if constexpr (MD % 2 == 0) {
#pragma unroll
          for (int q = 0; q < MD / 2; ++q) {
            const float2 v2 = *(const float2 *)(vrow + 2 * q);
            vf[e][2 * q] = v2.x;
            vf[e][2 * q + 1] = v2.y;
          }
        } else {
#pragma unroll
          for (int md = 0; md < MD; ++md) vf[e][md] = vrow[md];
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int md = 0; md < MD; ++md) o[md] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[e][md], pr[e], o[md], 0, 0, 0);
    }
  };

  {
    f32x4 kr[PCS], vr[PCS];
    fetch(t_first, kr, vr);
    stage(0, kr, vr);
  }
  __syncthreads();
  for (int t = t_first; t <= t_last; ++t) {
    const int buf = (t - t_first) & 1;
    f32x4 kr[PCS], vr[PCS];
    const bool more = t < t_last;
    if (more) fetch(t + 1, kr, vr);
    compute(buf, t);
    if (more) stage(buf ^ 1, kr, vr);
    __syncthreads();
  }

  // ---- normalise and store: lane holds dims (D/16) (4 kg + i) + md of its column ----
  const float l = xor32_sum(xor16_sum(lsum));
  if (!colok) return;
  const float inv = 1.f / l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const long d0 = qrow + MD * (4 * kg + i);
    if constexpr (DT == DD_F32 && MD % 4 == 0) {
#pragma unroll
      for (int q = 0; q < MD / 4; ++q)
        *(f32x4 *)((float *)p.out + d0 + 4 * q) =
            f32x4{o[4 * q][i], o[4 * q + 1][i], o[4 * q + 2][i], o[4 * q + 3][i]} * inv;
    } else {
#pragma unroll
      for (int md = 0; md < MD; ++md) store_as<DT>(p.out, d0 + md, o[md][i] * inv);
    }
  }
}

}  // namespace
