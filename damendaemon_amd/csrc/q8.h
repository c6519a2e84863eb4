// Q8_0 quantisation of one channel group (damendaemon/kv_quant.py:55-64).
#pragma once
#include "common.h"

// Quantises x[base .. base+group) into q[0 .. group) and returns the fp16
// scale bits.  scale = fp16(absmax / 127); inv = 0 for a zero scale, else
// 1 / float(scale); q = clamp(sign(y) * floor(|y| + 0.5), +-127), y = x*inv.
// Both divisions are done in double and rounded once to float, which gives
// the correctly rounded fp32 quotient (53 >= 2*24 + 2 bits), so the result
// is bit-identical to fp32 torch arithmetic whatever the fp32 divide mode.
template <int DT>
DD_DEV unsigned short q8_group(const void *x, long base, int group, signed char *q) {
  float amax = 0.f;
  for (int i = 0; i < group; ++i) amax = fmaxf(amax, fabsf(load_as<DT>(x, base + i)));
  const unsigned short sbits = float_to_f16_bits((float)((double)amax / 127.0));
  const float s = half_bits_to_float(sbits);
  const float inv = s == 0.f ? 0.f : (float)(1.0 / (double)s);
  for (int i = 0; i < group; ++i) {
    const float y = load_as<DT>(x, base + i) * inv;
    const float r = fminf(floorf(fabsf(y) + 0.5f), 127.f);
    q[i] = (signed char)(y < 0.f ? -r : r);
  }
  return sbits;
}

// ---- eight channels per lane -----------------------------------------------
// The kernels below give 8 consecutive channels (16 bytes of a 16-bit row) to
// a lane and 2^shift lanes to a channel group (the group's size / 8 rounded
// up to a power of two; lanes past the group hold zeros), so that a wave
// reads and writes whole rows.  One thread per group read its row at a stride
// of group * element size between lanes and touched every cache line once per
// element: 116 us for 4,160 tokens of 2 x 8 x 128 bf16 channels (0.2 TB/s);
// 9.1 us here (2.7 TB/s; launch and one memory round trip).

// The lane layout takes groups that are multiples of 8 up to 512 channels (64
// lanes), and rows that start on 16 bytes; returns the shift, or -1.
static inline int q8_lane_shift(int group) {
  if (group % 8 || group > 512) return -1;
  int shift = 0;
  while ((8 << shift) < group) ++shift;
  return shift;
}

// Channels idx .. idx + 7 of x (16-byte aligned), widened to fp32.
template <int DT>
DD_DEV void q8_load8(const void *x, long idx, float (&v)[8]) {
  if constexpr (DT == DD_F32) {
    const f32x4 a = *(const f32x4 *)((const float *)x + idx), b = *(const f32x4 *)((const float *)x + idx + 4);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = a[k];
      v[k + 4] = b[k];
    }
  } else {
    const u32x4 w = *(const u32x4 *)((const unsigned short *)x + idx);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[2 * k] = DT == DD_BF16 ? bf16_lo(w[k]) : f16_lo(w[k]);
      v[2 * k + 1] = DT == DD_BF16 ? bf16_hi(w[k]) : f16_hi(w[k]);
    }
  }
}

// q8_group over the 2^shift lanes of a group: this lane's eight codes, and
// the group's scale bits in every lane of it.  The same operations on every
// value as q8_group (the maximum is taken in another order, which changes
// nothing); the fp32 divisions are correctly rounded (this compiler's default
// for HIP, subnormal quotients included), which is what the roundings of the
// double quotients there give, at a tenth of their instructions.
DD_DEV u32x2 q8_lanes(const float (&v)[8], int shift, unsigned short *scale) {
#pragma clang fp contract(off)
  float amax = 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k) amax = fmaxf(amax, fabsf(v[k]));
  for (int off = (1 << shift) >> 1; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
  const unsigned short sbits = float_to_f16_bits(amax / 127.f);
  const float s = half_bits_to_float(sbits);
  const float inv = s == 0.f ? 0.f : 1.f / s;
  u32x2 codes = {0, 0};
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float y = v[k] * inv;
    const float r = fminf(floorf(fabsf(y) + 0.5f), 127.f);
    codes[k >> 2] |= ((unsigned)(int)(y < 0.f ? -r : r) & 0xffu) << (8 * (k & 3));
  }
  *scale = sbits;
  return codes;
}
