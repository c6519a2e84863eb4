// Fused rotary embedding + K/V page write (damendaemon/kernels.py:271-340).
//
// For token b and head h of the packed (T, (H + 2KH) * D) projection:
//   * query and key heads: optional RMS norm with a learned weight
//     (QK-norm), then rotate-half RoPE over the first RD channels:
//       out[j] = x[j]*cos[pos, j] + sgn(j) * x[(j + RD/2) % RD]*sin[pos, j]
//     with sgn = -1 for j < RD/2; channels j >= RD pass through (cos 1, sin 0);
//   * queries go to query[b, h, 0, :]; rotated keys and raw values go to the
//     cache row of position pos: page table[slot, pos / P], row pos % P (paged)
//     or slot / position (slotted); `materialize` also writes them densely.
// Without `precise`, the reference rounds to fp16 after each of the norm's
// two multiplies and after each of the two rotation products; every product
// and sum here is a separate correctly-rounded fp32 operation (no FMA
// contraction), as in the reference's enable_fp_fusion=False build.
//
// Two kernels.  rope_vec_kernel, for rows and cache of one dtype at head sizes
// that are multiples of 8 up to 512 and rotary widths that are multiples of
// 16: one workgroup per token (small batches: one per token and pass over
// the heads), so the position, slot and page lookups are done once
// per token; a lane owns 8 consecutive channels of a head (16-byte loads and
// stores), and the rotate-half partner channels come from the lane RD/16 away
// within the head's lane group.  rope_kernel, for everything else (mixed
// dtypes, odd sizes, rows that do not start on 16 bytes): one wavefront per
// (token, head), lanes striding over the channels.  Both apply
// the same per-element sequence of fp32 operations and fp16 roundings.
//
// Both are bound by memory.  Rotation of 2,462 fp32 tokens (32 + 8 heads of
// 128 channels, 121 MB with the cache rows): rope_kernel 56 us, which also
// reads every channel twice, 21.8 here.
#include "common.h"

// Every fp16 rounding below takes an fp32 value that has already been
// rounded: the reference rounds a product to fp32 and then to fp16, and the
// compiler would otherwise fold "fp32 multiply, then convert to fp16" into
// one mixed-precision FMA (v_fma_mix*) that rounds the exact product once --
// a different result whenever the fp32 product is an fp16 tie.
#pragma clang fp contract(off)

namespace {

DD_DEV float load_code(const void *p, long i, int code) {
  switch (code) {
    case DD_F32: return load_as<DD_F32>(p, i);
    case DD_F16: return load_as<DD_F16>(p, i);
    default: return load_as<DD_BF16>(p, i);
  }
}

DD_DEV float round_f16(float x) {
  asm("" : "+v"(x));   // x is an fp32 value here, not an expression the conversion may absorb
  return half_bits_to_float(float_to_f16_bits(x));
}

struct RopeParams {
  const void *x;
  const void *cos;
  const void *sin;
  const int64_t *pos;
  const int64_t *slots;
  const void *qw;
  const void *kw;
  const int32_t *table;
  void *q;
  void *ck;
  void *cv;
  void *tk;
  void *tv;
  long tokens;
  long capacity;
  int H, KH, D, RD;
  int C;  // page size (paged) or context (slotted)
  int table_w, table_rows;
  int cos_code, w_code;
  int lane_shift;  // rope_vec_kernel: 2^lane_shift lanes per head
  int precise;
  float eps;
};

template <int XT, int CT>
__global__ __launch_bounds__(256) void rope_kernel(RopeParams p) {
  const int lane = threadIdx.x & 63;
  const long item = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int heads = p.H + 2 * p.KH;
  if (item >= p.tokens * heads) return;
  const long b = item / heads;
  const int head = (int)(item - b * heads);
  const long pos = p.pos[b];
  const long slot = p.slots[b];
  long cslot = slot, cpos = pos;
  if (p.table) {
    const long entry = pos / p.C;
    cslot = (slot >= 0 && slot < p.table_rows && entry < p.table_w) ? p.table[slot * p.table_w + entry] : -1;
    cpos = pos % p.C;
  }
  const bool cache_ok = cslot >= 0 && cslot < p.capacity;
  const long base = (b * heads + head) * (long)p.D;
  const int D = p.D, RD = p.RD, half = RD / 2;

  if (head >= p.H + p.KH) {  // value head: stored as is
    const int kh = head - p.H - p.KH;
    for (int j = lane; j < D; j += 64) {
      const float x = load_as<XT>(p.x, base + j);
      if (cache_ok) store_as<CT>(p.cv, ((cslot * p.KH + kh) * p.C + cpos) * D + j, x);
      if (p.tv) store_as<CT>(p.tv, (b * p.KH + kh) * (long)D + j, x);
    }
    return;
  }
  const bool is_q = head < p.H;
  const void *w = is_q ? p.qw : p.kw;
  float inv = 1.f;
  if (w) {
    float ss = 0.f;
    for (int j = lane; j < D; j += 64) {
      const float x = load_as<XT>(p.x, base + j);
      ss += x * x;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    inv = 1.f / sqrtf(__fadd_rn(ss / (float)D, p.eps));
  }
  for (int j = lane; j < D; j += 64) {
    const int oj = (j + half) % RD;
    float x = load_as<XT>(p.x, base + j);
    float o = load_as<XT>(p.x, base + oj);
    if (w) {
      x = __fmul_rn(x, inv);
      o = __fmul_rn(o, inv);
      if (!p.precise) { x = round_f16(x); o = round_f16(o); }
      x = __fmul_rn(x, load_code(w, j, p.w_code));
      o = __fmul_rn(o, load_code(w, oj, p.w_code));
      if (!p.precise) { x = round_f16(x); o = round_f16(o); }
    }
    if (j < half) o = -o;
    const float c = j < RD ? load_code(p.cos, pos * RD + j, p.cos_code) : 1.f;
    const float s = j < RD ? load_code(p.sin, pos * RD + j, p.cos_code) : 0.f;
    float a = __fmul_rn(x, c);
    float bb = __fmul_rn(o, s);
    if (!p.precise) { a = round_f16(a); bb = round_f16(bb); }
    const float r = __fadd_rn(a, bb);
    if (is_q) {
      store_as<XT>(p.q, (b * p.H + head) * (long)D + j, r);
    } else {
      const int kh = head - p.H;
      if (cache_ok) store_as<CT>(p.ck, ((cslot * p.KH + kh) * p.C + cpos) * D + j, r);
      if (p.tk) store_as<CT>(p.tk, (b * p.KH + kh) * (long)D + j, r);
    }
  }
}

// 16-bit <-> fp32 for the 16-bit row formats (bit patterns in the low half)
template <int XT>
DD_DEV float h2f(unsigned h) {
  if constexpr (XT == DD_BF16) return __uint_as_float(h << 16);
  else return half_bits_to_float((unsigned short)h);
}
template <int XT>
DD_DEV unsigned f2h(float x) {
  if constexpr (XT == DD_BF16) return float_to_bf16_bits(x);
  else return float_to_f16_bits(x);
}

// Eight consecutive values (16-byte aligned) as fp32, and back.
template <int DT, int N>
DD_DEV void rope_widen8(const u32x4 (&w)[N], float (&v)[8]) {
  if constexpr (DT == DD_F32) {
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = __uint_as_float(w[k >> 2][k & 3]);
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[2 * k] = h2f<DT>(w[0][k] & 0xffffu);
      v[2 * k + 1] = h2f<DT>(w[0][k] >> 16);
    }
  }
}
template <int DT>
DD_DEV void rope_load8(const void *p, long i, float (&v)[8]) {
  constexpr int N = DT == DD_F32 ? 2 : 1;
  const u32x4 *src = (const u32x4 *)((const char *)p + (DT == DD_F32 ? 4 : 2) * i);
  u32x4 w[N];
#pragma unroll
  for (int q = 0; q < N; ++q) w[q] = src[q];
  rope_widen8<DT>(w, v);
}
DD_DEV void rope_load8_code(const void *p, long i, int code, float (&v)[8]) {
  switch (code) {
    case DD_F32: rope_load8<DD_F32>(p, i, v); break;
    case DD_F16: rope_load8<DD_F16>(p, i, v); break;
    default: rope_load8<DD_BF16>(p, i, v); break;
  }
}
template <int DT>
DD_DEV void rope_store8(void *p, long i, const float (&v)[8]) {
  if constexpr (DT == DD_F32) {
    *(f32x4 *)((float *)p + i) = f32x4{v[0], v[1], v[2], v[3]};
    *(f32x4 *)((float *)p + i + 4) = f32x4{v[4], v[5], v[6], v[7]};
  } else {
    u32x4 r;
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = f2h<DT>(v[2 * k]) | (f2h<DT>(v[2 * k + 1]) << 16);
    *(u32x4 *)((unsigned short *)p + i) = r;
  }
}

// Norm (when wt is set) and rotation of one head's eight channels of a lane.
// Plain operators: under this file's pragma they are not contracted, while the
// __fmul_rn / __fadd_rn of the headers, compiled before it, are where nothing
// stands between them.
template <bool PRECISE>
DD_DEV void rope_rotate(const RopeParams &p, const void *wt, int shift, int j0, bool on, int partner, bool lower,
                        const float (&c)[8], const float (&sn)[8], float (&x)[8], float (&r)[8]) {
  auto rnd = [](float v) { return PRECISE ? v : round_f16(v); };
  if (wt) {
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) ss += x[k] * x[k];
    for (int off = (1 << shift) >> 1; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    const float inv = 1.f / sqrtf(ss / (float)p.D + p.eps);
    float wv[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (on) rope_load8_code(wt, j0, p.w_code, wv);
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = rnd(rnd(x[k] * inv) * wv[k]);
  }
  float o[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) o[k] = shfl(x[k], partner);
#pragma unroll
  for (int k = 0; k < 8; ++k)
    r[k] = rnd(x[k] * c[k]) + rnd((lower ? -o[k] : o[k]) * sn[k]);
}

// FULL: full-width rotation of a power-of-two head, so that every lane has
// channels to rotate and none of the other shapes' conditions is needed.
#ifndef DD_ROPE_PASSES
#define DD_ROPE_PASSES 4
#endif
template <int XT, int CS, bool FULL>
__global__ __launch_bounds__(256) void rope_vec_kernel(RopeParams p) {
  constexpr int N = XT == DD_F32 ? 2 : 1;    // 16-byte pieces of eight channels
  constexpr int ES = XT == DD_F32 ? 4 : 2;   // bytes per element
  constexpr int kPasses = DD_ROPE_PASSES;
  const long b = blockIdx.x;
  const int D = p.D, RD = p.RD;
  const int shift = p.lane_shift;        // 2^shift lanes per head, D / 8 of them with channels
  const int hl = threadIdx.x & ((1 << shift) - 1);   // lane within the head's group
  const int hpp = 256 >> shift;          // heads per pass of the workgroup
  const int heads = p.H + 2 * p.KH;
  const long pos = p.pos[b];
  const long slot = p.slots[b];
  long cslot = slot, cpos = pos;
  if (p.table) {
    // (32-bit division where the position allows: the 64-bit one is a long sequence)
    const long entry = (unsigned long)pos <= 0xffffffffUL ? (long)((unsigned)pos / (unsigned)p.C) : pos / p.C;
    cslot = (slot >= 0 && slot < p.table_rows && entry < p.table_w) ? p.table[slot * p.table_w + entry] : -1;
    cpos = pos - entry * p.C;
  }
  const bool cache_ok = cslot >= 0 && cslot < p.capacity;
  const int j0 = 8 * hl;
  const bool on = FULL || j0 < D;        // (idle lanes stay for the shuffles, with zeros)
  // cos / sin of this lane's channels at the token's position; 1 and 0 past
  // the rotary width
  float c[8], sn[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    c[k] = 1.f;
    sn[k] = 0.f;
  }
  if (FULL || j0 < RD) {
    rope_load8<CS>(p.cos, pos * RD + j0, c);
    rope_load8<CS>(p.sin, pos * RD + j0, sn);
  }
  const bool lower = j0 < RD / 2;        // channels below RD / 2: the partner enters negated
  // lane of channel (j0 + RD / 2) % RD
  const int lane = threadIdx.x & 63;
  const int partner = FULL ? lane ^ (1 << shift >> 1) : lane - hl + (hl + RD / 16) % (RD / 8);
  const int stride = hpp * (int)gridDim.y;
  // kPasses heads' rows in flight per lane: every load of a batch goes out
  // before any of its stores (the compiler orders a load behind the stores
  // issued before it, so one row at a time waited for a full round trip each)
  for (int h0 = (int)(blockIdx.y * hpp + (threadIdx.x >> shift)); h0 < heads; h0 += kPasses * stride) {
    u32x4 raw[kPasses][N];
#pragma unroll
    for (int u = 0; u < kPasses; ++u) {
      const int h = min(h0 + u * stride, heads - 1);   // (clamped: loads behind no branch)
      const u32x4 *src = (const u32x4 *)((const char *)p.x + ES * ((b * heads + h) * (long)D + (on ? j0 : 0)));
#pragma unroll
      for (int q = 0; q < N; ++q) raw[u][q] = src[q];
    }
#pragma unroll
    for (int u = 0; u < kPasses; ++u) {
      const int h = h0 + u * stride;
      if (h >= heads) break;
      const bool is_q = h < p.H, is_v = h >= p.H + p.KH;
      const int kh = h - (is_v ? p.H + p.KH : p.H);
      const long row = is_q ? (b * p.H + h) * (long)D + j0 : ((cslot * p.KH + kh) * p.C + cpos) * D + j0;
      const long dense = (b * p.KH + kh) * (long)D + j0;
      if (is_v) {  // value head: stored as is
        if (!on) continue;
#pragma unroll
        for (int q = 0; q < N; ++q) {
          if (cache_ok) ((u32x4 *)((char *)p.cv + ES * row))[q] = raw[u][q];
          if (p.tv) ((u32x4 *)((char *)p.tv + ES * dense))[q] = raw[u][q];
        }
        continue;
      }
      float x[8];
      rope_widen8<XT>(raw[u], x);
      if constexpr (!FULL) {
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = on ? x[k] : 0.f;   // (lanes past the head: nothing in the norm's sum)
      }
      float r[8];
      if (p.precise)
        rope_rotate<true>(p, is_q ? p.qw : p.kw, shift, j0, on, partner, lower, c, sn, x, r);
      else
        rope_rotate<false>(p, is_q ? p.qw : p.kw, shift, j0, on, partner, lower, c, sn, x, r);
      if (!on) continue;
      if (is_q) {
        rope_store8<XT>(p.q, row, r);
      } else {
        if (cache_ok) rope_store8<XT>(p.ck, row, r);
        if (p.tk) rope_store8<XT>(p.tk, dense, r);
      }
    }
  }
}

template <int XT>
int launch_rope_vec(RopeParams p, hipStream_t s) {
  if (p.tokens > 0x7fffffffL) return DD_EUNSUPPORTED;
  p.lane_shift = 0;
  while ((8 << p.lane_shift) < p.D) ++p.lane_shift;
  // With few tokens (fewer workgroups than CUs) the passes over the heads run
  // as workgroups of their own; with many, one workgroup per token is faster
  // (4,216 tokens, bf16: 25 us against 31).
  const long passes = dd_cdiv(p.H + 2 * p.KH, 256 >> p.lane_shift);
  const dim3 grid((unsigned)p.tokens, p.tokens <= 256 ? (unsigned)(passes < 64 ? passes : 64) : 1u);
  const bool full = p.RD == p.D && (8 << p.lane_shift) == p.D && p.D >= 16;
#define DD_ROPE_VEC(CS)                                                                                      \
  if (full) hipLaunchKernelGGL((rope_vec_kernel<XT, CS, true>), grid, dim3(256), 0, s, p);                  \
  else hipLaunchKernelGGL((rope_vec_kernel<XT, CS, false>), grid, dim3(256), 0, s, p)
  switch (p.cos_code) {
    case DD_F32: DD_ROPE_VEC(DD_F32); break;
    case DD_F16: DD_ROPE_VEC(DD_F16); break;
    case DD_BF16: DD_ROPE_VEC(DD_BF16); break;
    default: return DD_EUNSUPPORTED;
  }
#undef DD_ROPE_VEC
  DD_LAUNCH_CHECK();
  return DD_OK;
}

template <int XT>
int launch_rope(const RopeParams &p, int ct, hipStream_t s) {
  const long items = p.tokens * (p.H + 2 * p.KH);
  const dim3 grid((unsigned)dd_cdiv(items, 4));
  switch (ct) {
    case DD_F32: hipLaunchKernelGGL((rope_kernel<XT, DD_F32>), grid, dim3(256), 0, s, p); break;
    case DD_F16: hipLaunchKernelGGL((rope_kernel<XT, DD_F16>), grid, dim3(256), 0, s, p); break;
    case DD_BF16: hipLaunchKernelGGL((rope_kernel<XT, DD_BF16>), grid, dim3(256), 0, s, p); break;
    default: return DD_EUNSUPPORTED;
  }
  DD_LAUNCH_CHECK();
  return DD_OK;
}

}  // namespace

extern "C" int dd_rope_batch(const void *qkv, int qkv_dtype, const void *cos, const void *sin, int cos_dtype,
                             int rotary_dim, const int64_t *positions, const int64_t *slots, int64_t tokens,
                             int heads, int kv_heads, int dim, const void *q_norm, const void *k_norm,
                             int norm_dtype, float eps, int precise, const int32_t *page_table, int table_rows,
                             int table_width, void *query, void *cache_k, void *cache_v, int cache_dtype,
                             int64_t capacity, int cache_len, void *key_out, void *value_out, void *stream) {
  if (!qkv || !cos || !sin || !positions || !slots || !query || !cache_k || !cache_v || tokens < 0 ||
      heads <= 0 || kv_heads <= 0 || dim <= 0 || rotary_dim <= 0 || rotary_dim > dim || rotary_dim % 2 ||
      cache_len <= 0 || capacity <= 0 || ((q_norm || k_norm) && rotary_dim != dim))
    return DD_EINVAL;
  if (tokens == 0) return DD_OK;
  RopeParams p{};
  p.x = qkv;
  p.cos = cos;
  p.sin = sin;
  p.pos = positions;
  p.slots = slots;
  p.qw = q_norm;
  p.kw = k_norm;
  p.table = page_table;
  p.q = query;
  p.ck = cache_k;
  p.cv = cache_v;
  p.tk = key_out;
  p.tv = value_out;
  p.tokens = tokens;
  p.capacity = capacity;
  p.H = heads;
  p.KH = kv_heads;
  p.D = dim;
  p.RD = rotary_dim;
  p.C = cache_len;
  p.table_w = table_width;
  p.table_rows = table_rows;
  p.cos_code = cos_dtype;
  p.w_code = norm_dtype;
  p.precise = precise;
  p.eps = eps;
  hipStream_t s = (hipStream_t)stream;
  // the 16-byte accesses of the vector kernel need 16-byte aligned rows
  auto a16 = [](const void *q) { return dd_aligned(q, 16); };
  const bool aligned = a16(qkv) && a16(cos) && a16(sin) && a16(query) && a16(cache_k) && a16(cache_v) &&
                       a16(key_out) && a16(value_out) && a16(q_norm) && a16(k_norm);
  // Rows of whole 16-byte pieces whose rotate-half partners are whole pieces
  // too (the rotary width a multiple of 16), a head within one wave, and no
  // conversion between rows and cache.  (The vector kernel was built for
  // full-width rotation of 16-bit rows at 64 / 128 / 256 first; at the
  // other sizes and in fp32 rope_kernel took 2 to 4 times its time.)
  if (aligned && dim % 8 == 0 && dim <= 512 && rotary_dim % 16 == 0 && cache_dtype == qkv_dtype) {
    if (qkv_dtype == DD_F32) return launch_rope_vec<DD_F32>(p, s);
    if (qkv_dtype == DD_BF16) return launch_rope_vec<DD_BF16>(p, s);
    if (qkv_dtype == DD_F16) return launch_rope_vec<DD_F16>(p, s);
  }
  switch (qkv_dtype) {
    case DD_F32: return launch_rope<DD_F32>(p, cache_dtype, s);
    case DD_F16: return launch_rope<DD_F16>(p, cache_dtype, s);
    case DD_BF16: return launch_rope<DD_BF16>(p, cache_dtype, s);
    default: return DD_EUNSUPPORTED;
  }
}
