// Q8_0 KV codec (damendaemon/kv_quant.py:48-76) for gfx950.
//
// Per group of `group` consecutive channels of a row:
//   scale = fp16(absmax / 127)                       (fp32 divide, RNE to fp16)
//   inv   = scale == 0 ? 0 : 1 / float(scale)        (correctly rounded)
//   q     = clamp(sign(x*inv) * floor(|x*inv| + 0.5), -127, 127)
// Dequantisation is int8 * float(scale), rounded once to the output dtype.
// Every step is a single correctly-rounded fp32 operation, so the result is
// bit-identical to the reference's torch arithmetic.  The two divisions are
// done in double and rounded once to float, which yields the correctly
// rounded fp32 quotient (53 >= 2*24+2 bits), independent of the compiler's
// fp32 division mode.
//
// Eight channels per lane, a channel group across lanes (q8.h); groups that
// are not multiples of 8 channels, or larger than 512, and rows that do not
// start on 16 bytes take one thread per group (quantise) or channel
// (dequantise).
#include "common.h"
#include "q8.h"

namespace {

template <int DT>
__global__ __launch_bounds__(256) void quantize_kernel(const void *x, long groups, int group,
                                                       signed char *q, unsigned short *scale) {
  const long g = (long)blockIdx.x * 256 + threadIdx.x;
  if (g >= groups) return;
  scale[g] = q8_group<DT>(x, g * group, group, q + g * group);
}

template <int DT>
__global__ __launch_bounds__(256) void dequantize_kernel(const signed char *q, const unsigned short *scale,
                                                         long n, int group, void *out) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  store_as<DT>(out, i, (float)q[i] * half_bits_to_float(scale[i / group]));
}

// 2^shift lanes per group, 8 channels per lane; n = groups << shift lanes.
template <int DT>
__global__ __launch_bounds__(256) void quantize_lanes_kernel(const void *x, long n, int group, int shift,
                                                             signed char *q, unsigned short *scale) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  const long g = i >> shift;
  const int c = 8 * (int)(i & ((1 << shift) - 1));
  const bool on = i < n && c < group;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (on) q8_load8<DT>(x, g * group + c, v);
  unsigned short sbits;
  const u32x2 codes = q8_lanes(v, shift, &sbits);
  if (on) *(u32x2 *)(q + g * group + c) = codes;
  if (on && c == 0) scale[g] = sbits;
}

// Eight channels per thread: 8 bytes of codes, one scale, 16 or 32 bytes out.
template <int DT>
__global__ __launch_bounds__(256) void dequantize_lanes_kernel(const signed char *q, const unsigned short *scale,
                                                               long n8, int group8, void *out) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  // (32-bit division where it suffices: the 64-bit one is a long sequence)
  const long g = n8 <= 0xffffffffL ? (long)((unsigned)i / (unsigned)group8) : i / group8;
  const u32x2 w = ((const u32x2 *)q)[i];
  const float s = half_bits_to_float(scale[g]);
  float y[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) y[k] = (float)(int)(signed char)(w[k >> 2] >> (8 * (k & 3))) * s;
  if constexpr (DT == DD_F32) {
    ((f32x4 *)out)[2 * i] = f32x4{y[0], y[1], y[2], y[3]};
    ((f32x4 *)out)[2 * i + 1] = f32x4{y[4], y[5], y[6], y[7]};
  } else {
    u32x4 r;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const unsigned lo = DT == DD_BF16 ? float_to_bf16_bits(y[2 * k]) : float_to_f16_bits(y[2 * k]);
      const unsigned hi = DT == DD_BF16 ? float_to_bf16_bits(y[2 * k + 1]) : float_to_f16_bits(y[2 * k + 1]);
      r[k] = lo | (hi << 16);
    }
    ((u32x4 *)out)[i] = r;
  }
}

}  // namespace

extern "C" int dd_quantize_q8(const void *x, int x_dtype, int64_t rows, int dim, int group, void *q, void *scale,
                              void *stream) {
  if (!x || !q || !scale || rows < 0 || dim <= 0 || group <= 0 || dim % group) return DD_EINVAL;
  const long groups = rows * (long)(dim / group);
  if (groups == 0) return DD_OK;
  hipStream_t s = (hipStream_t)stream;
  auto *qq = (signed char *)q;
  auto *ss = (unsigned short *)scale;
  const int shift = q8_lane_shift(group);
  if (shift >= 0 && dd_aligned(x, 16) && dd_aligned(q, 8) && groups <= (0x7fffffffL << 8 >> shift)) {
    const long n = groups << shift;
    const dim3 lanes((unsigned)dd_cdiv(n, 256));
    switch (x_dtype) {
      case DD_F32: hipLaunchKernelGGL(quantize_lanes_kernel<DD_F32>, lanes, dim3(256), 0, s, x, n, group, shift, qq, ss); break;
      case DD_F16: hipLaunchKernelGGL(quantize_lanes_kernel<DD_F16>, lanes, dim3(256), 0, s, x, n, group, shift, qq, ss); break;
      case DD_BF16: hipLaunchKernelGGL(quantize_lanes_kernel<DD_BF16>, lanes, dim3(256), 0, s, x, n, group, shift, qq, ss); break;
      default: return DD_EUNSUPPORTED;
    }
    DD_LAUNCH_CHECK();
    return DD_OK;
  }
  const dim3 grid((unsigned)dd_cdiv(groups, 256));
  switch (x_dtype) {
    case DD_F32: hipLaunchKernelGGL(quantize_kernel<DD_F32>, grid, dim3(256), 0, s, x, groups, group, qq, ss); break;
    case DD_F16: hipLaunchKernelGGL(quantize_kernel<DD_F16>, grid, dim3(256), 0, s, x, groups, group, qq, ss); break;
    case DD_BF16: hipLaunchKernelGGL(quantize_kernel<DD_BF16>, grid, dim3(256), 0, s, x, groups, group, qq, ss); break;
    default: return DD_EUNSUPPORTED;
  }
  DD_LAUNCH_CHECK();
  return DD_OK;
}

extern "C" int dd_dequantize_q8(const void *q, const void *scale, int64_t rows, int dim, int group, void *out,
                                int out_dtype, void *stream) {
  if (!q || !scale || !out || rows < 0 || dim <= 0 || group <= 0 || dim % group) return DD_EINVAL;
  const long n = rows * (long)dim;
  if (n == 0) return DD_OK;
  hipStream_t s = (hipStream_t)stream;
  auto *qq = (const signed char *)q;
  auto *ss = (const unsigned short *)scale;
  if (group % 8 == 0 && dd_aligned(q, 8) && dd_aligned(out, 16)) {
    const long n8 = n / 8;
    const dim3 lanes((unsigned)dd_cdiv(n8, 256));
    switch (out_dtype) {
      case DD_F32: hipLaunchKernelGGL(dequantize_lanes_kernel<DD_F32>, lanes, dim3(256), 0, s, qq, ss, n8, group / 8, out); break;
      case DD_F16: hipLaunchKernelGGL(dequantize_lanes_kernel<DD_F16>, lanes, dim3(256), 0, s, qq, ss, n8, group / 8, out); break;
      case DD_BF16: hipLaunchKernelGGL(dequantize_lanes_kernel<DD_BF16>, lanes, dim3(256), 0, s, qq, ss, n8, group / 8, out); break;
      default: return DD_EUNSUPPORTED;
    }
    DD_LAUNCH_CHECK();
    return DD_OK;
  }
  const dim3 grid((unsigned)dd_cdiv(n, 256));
  switch (out_dtype) {
    case DD_F32: hipLaunchKernelGGL(dequantize_kernel<DD_F32>, grid, dim3(256), 0, s, qq, ss, n, group, out); break;
    case DD_F16: hipLaunchKernelGGL(dequantize_kernel<DD_F16>, grid, dim3(256), 0, s, qq, ss, n, group, out); break;
    case DD_BF16: hipLaunchKernelGGL(dequantize_kernel<DD_BF16>, grid, dim3(256), 0, s, qq, ss, n, group, out); break;
    default: return DD_EUNSUPPORTED;
  }
  DD_LAUNCH_CHECK();
  return DD_OK;
}
