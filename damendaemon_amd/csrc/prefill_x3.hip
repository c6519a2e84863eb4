// Chunked-prefill attention over fp32 pages with fp32-accurate products on the
// bf16 matrix cores (gfx950), head sizes that are multiples of 16 up to 128.
//
// Semantics as in the other prefill kernels (damendaemon/paged.py:97-111 with
// qwen2.py:754-770): query row j of segment i attends keys 0 .. start_i + j of
// its slot (and > position - window), GQA head h reads KV head h / G,
// softmax(q.k * scale) . v.
//
// Products.  An fp32 value is the sum of three bf16 values exactly: its own
// rounding, the rounding of what is left, and the rest (8 + 8 + 8 bits).  Of
// the nine products of two such sums the six of weight 2^-18 and above are
// formed, each exact in the matrix core's fp32 accumulation; the three that
// are left out are below 2^-26 of the product, a quarter of the rounding that
// an fp32 product of its own would get.  The error against 64 bits is no
// larger than v_mfma_f32's (2-norm over 2,462 rows of 32 heads of 128, rotated
// keys included: 7.0e-7 of the result against 9.3e-7), at 16 / 6 of its rate.
// What the parts cannot hold: a value past bf16's range (above 3.39e38, or
// infinite) gives a non-finite result, and parts below 2^-126 are lost, which
// shows where a whole result is below 2^-100 or the queries are that small (or
// so large that a key's lost part counts).  Items with such outputs or queries
// flag themselves, and the workgroup recomputes them with fp32 matrix
// instructions (prefill_f32_item.h; another launch where keys are split).
//
// Work split.  Bound by the matrix cores: a workgroup of eight waves (two per
// SIMD, one workgroup per CU) owns 256 (query row, head) columns of one
// (segment, KV head), 32 per wave, with Q's three parts in registers; keys
// come in 32-key tiles.  Every thread loads one 8-dim piece of a K and of a V
// row (plain loads, in flight during the P.V products of the tile before),
// splits it and writes the parts to LDS, so a tile is read and split once for
// the whole workgroup; two LDS buffers, one barrier per tile.  Per tile and
// wave 2 x 3 D / 8 MFMAs (32x32x16) against ~150 vector operations of softmax
// and splitting.  8 x 512 fp32 tokens on contexts up to 4,608, 32 / 8 heads of
// 128: 2,330 us on the fp32 matrix cores (83 TFLOP/s), 1,036 us here (187; 1,125
// on the bf16 ones); 96 dims 1,747 -> 825 us, 64 dims 1,189 -> 580 us.
//
// LDS layouts.  K part: block of 8 dims x 32 keys, 16 bytes per key, 576 bytes
// per block (64 of padding: the eight lanes of a write phase, four keys of two
// blocks, hit distinct banks); an S^T operand read is two runs of 512
// contiguous bytes.  V part: the regions of prefill_pipe.hip, which the
// transposing read hands out in the order of the S^T accumulator, so that P^T
// is a slice of it.
//
// Few work items for the chip: the keys are split over workgroups as in
// prefill_pipe.hip and combined by prefill_merge_kernel.
#include "prefill_generic.h"
#include "prefill_merge.h"

#include <climits>

namespace dd_prefill {
namespace {

constexpr int kX3Waves = 8;
constexpr int kX3Keys = DD_PREFILL_X3_KEYS;   // keys per tile
constexpr int kKBlock = 576;                  // bytes of one 8-dim block of a K part

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// The three bf16 parts of a and b, packed in pairs.
DD_DEV void split3(float a, float b, unsigned &h, unsigned &m, unsigned &l) {
  h = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
  a -= __uint_as_float(h << 16);
  b -= __uint_as_float(h & 0xffff0000u);
  m = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
  a -= __uint_as_float(m << 16);
  b -= __uint_as_float(m & 0xffff0000u);
  l = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
// Part j of eight values in r[j].
DD_DEV void split3(const f32x4 (&x)[2], u32x4 (&r)[3]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    unsigned h, m, l;
    split3(x[i >> 1][2 * (i & 1)], x[i >> 1][2 * (i & 1) + 1], h, m, l);
    r[0][i] = h;
    r[1][i] = m;
    r[2][i] = l;
  }
}

DD_DEV f32x16 mfma_bf16(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
}
// c += sum of the six products of parts a[i], b[j] with i + j <= 2, smallest first.
DD_DEV f32x16 mfma_x3(const u32x4 (&a)[3], const u32x4 (&b)[3], f32x16 c) {
  c = mfma_bf16(a[2], b[0], c);
  c = mfma_bf16(a[1], b[1], c);
  c = mfma_bf16(a[0], b[2], c);
  c = mfma_bf16(a[1], b[0], c);
  c = mfma_bf16(a[0], b[1], c);
  return mfma_bf16(a[0], b[0], c);
}

DD_DEV u32x2 lds_tr(const char *p) {
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(const lds_void *)p));
}

template <int D>
__global__ __launch_bounds__(64 * kX3Waves) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_x3_kernel(PrefillParams p) {
#if __HIP_DEVICE_COMPILE__
  static_assert(D % 16 == 0 && D <= 128, "head size");
  constexpr int NT = 64 * kX3Waves;
  constexpr int COLS = 32 * kX3Waves;
  constexpr int KT = kX3Keys;
  constexpr int NCC = D / 16;               // k-steps of S^T
  constexpr int MD = (D + 31) / 32;         // 32-dim blocks of O^T
  constexpr int PD = 4 * MD;                // 8-dim pieces of a row, the last block's missing dims included
  constexpr int KPART = D / 8 * kKBlock;    // bytes of one part of a K tile
  constexpr int VPART = 2048 * MD;          // ... of a V tile: (16-key step, dim block, half) regions of 512
  static_assert(KT == 32 && KT * PD <= NT, "one piece per thread");

  __shared__ __align__(16) char s_mem[6 * (KPART + VPART)];
  static_assert(f32_lds<D>() <= 6 * (KPART + VPART), "the fp32 re-run fits");
  // [2][3 parts] of K, then of V
  auto s_k = [&](int buf) __attribute__((always_inline)) { return s_mem + buf * 3 * KPART; };
  auto s_v = [&](int buf) __attribute__((always_inline)) { return s_mem + 6 * KPART + buf * 3 * VPART; };
  __shared__ int s_flag;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = uniform(tid >> 6);
  const int l32 = lane & 31;
  const int h2 = lane >> 5;

  PrefillItem it;
  if (!prefill_item<false>(p, it, 0)) return;
  const int G = p.G;
  const int rows = COLS / G;
  const int r0 = it.qt * rows;
  if (r0 >= it.len) return;
  const int rows_here = min(rows, it.len - r0);
  const int kh = it.grp - it.seg * p.KH;
  int t_first, t_last;
  const int nsplit = prefill_tiles<true>(p, it, KT, r0, rows_here, t_first, t_last);
  if (it.split >= nsplit) return;
  const int context = it.start + it.len;

  // ---- this lane's column and its Q^T operands ----
  const int col = w * 32 + l32;
  const int qr = col / G;
  const int gh = col - qr * G;
  const bool colok = qr < rows_here;
  const int qpos = it.start + r0 + qr;
  const long qrow = ((it.tok0 + r0 + (colok ? qr : 0)) * p.H + (long)kh * G + gh) * D;
  u32x4 qa[NCC][3];
  float qmax = 0.f;   // the column's largest |q|
#pragma unroll
  for (int c = 0; c < NCC; ++c) {
    const f32x4 *src = (const f32x4 *)((const float *)p.q + qrow + 16 * c + 8 * h2);
    f32x4 x[2] = {src[0], src[1]};
#pragma unroll
    for (int i = 0; i < 2; ++i) x[i] = colok ? x[i] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 8; ++i) qmax = fmaxf(qmax, fabsf(x[i >> 2][i & 3]));
    split3(x, qa[c]);
  }
  qmax = xor32_max(qmax);
  const bool q_odd = qmax != 0.f && !(qmax >= 0x1p-60f && qmax <= 0x1p64f);   // (NaN queries are NaN rows anyway)

  // ---- tile staging: this thread's piece is key `pkey`, dims 8 pd ..+8 ----
  const int pd = (tid >> 2) % PD;
  const int pkey = 4 * ((tid >> 2) / PD) + (tid & 3);
  const bool piece = pkey < KT;
  const bool pload = piece && 8 * pd < D;
  const bool slot_ok = it.slot >= 0 && it.slot < p.table_rows;
  // page of this thread's key of tile t, or -1
  auto lookup = [&](int t) __attribute__((always_inline)) -> int {
    const int entry = (t * KT + pkey) >> p.page_shift;
    int phys = -1;
    if (pload && slot_ok && t <= t_last && entry < p.table_w) phys = p.table[it.slot * p.table_w + entry];
    return phys;
  };
  auto fetch = [&](int t, int phys, f32x4 (&kr)[2], f32x4 (&vr)[2]) __attribute__((always_inline)) {
    const int key = t * KT + pkey;
#pragma unroll
    for (int i = 0; i < 2; ++i) kr[i] = vr[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (phys >= 0 && phys < p.capacity && key < context) {
      const long base = ((((long)phys * p.KH + kh) << p.page_shift) + (key & (p.page - 1))) * (long)D + 8 * pd;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        kr[i] = ((const f32x4 *)((const float *)p.k + base))[i];
        vr[i] = ((const f32x4 *)((const float *)p.v + base))[i];
      }
    }
  };
  const int k_wr = pd * kKBlock + pkey * 16;
  const int v_wr = (((pkey >> 4) * MD + (pd >> 2)) * 2 + ((pkey >> 3) & 1)) * 512 +
                   8 * (32 * ((pkey >> 2) & 1) + 16 * ((pd >> 1) & 1) + 4 * (pkey & 3) + 2 * (pd & 1));
  auto stage = [&](int buf, const f32x4 (&kr)[2], const f32x4 (&vr)[2]) __attribute__((always_inline)) {
    u32x4 r[3];
    if (pload) {
      split3(kr, r);
#pragma unroll
      for (int j = 0; j < 3; ++j) *(u32x4 *)(s_k(buf) + j * KPART + k_wr) = r[j];
    }
    if (piece) {
      split3(vr, r);
#pragma unroll
      for (int j = 0; j < 3; ++j) *(u32x4 *)(s_v(buf) + j * VPART + v_wr) = r[j];
    }
  };

  f32x16 o[MD];
#pragma unroll
  for (int md = 0; md < MD; ++md) o[md] = f32x16{};
  float m_run = kNegInf;   // running offset of this lane's column (scaled, exp2 domain)
  float l_part = 0.f;      // this lane's share of the column's denominator

  const int k_rd = h2 * kKBlock + l32 * 16;
  f32x4 kr[2], vr[2];
  fetch(t_first, lookup(t_first), kr, vr);
  int phys = lookup(t_first + 1);
  if (tid == 0) s_flag = 0;
  stage(0, kr, vr);
  const int odd = __syncthreads_or(q_odd);
  for (int t = t_first; t <= t_last; ++t) {
    const int buf = (t - t_first) & 1;
    // ---- S^T = K Q^T ----
    f32x16 s = {};
#pragma unroll
    for (int c = 0; c < NCC; ++c) {
      u32x4 ka[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) ka[j] = *(const u32x4 *)(s_k(buf) + j * KPART + 2 * c * kKBlock + k_rd);
      s = mfma_x3(ka, qa[c], s);
    }
    // ---- softmax: register r holds key 32 t + 8 (r / 4) + 4 h2 + r % 4 ----
    const int kbase = t * KT;
    const bool whole = kbase + KT - 1 <= it.start + r0 &&
                       (p.window <= 0 || kbase >= it.start + r0 + rows_here - p.window);
    float mx = kNegInf;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] *= p.scale_log2;
      if (!whole) {
        const int key = kbase + 8 * (r >> 2) + 4 * h2 + (r & 3);
        s[r] = (key <= qpos) & ((p.window <= 0) | (key > qpos - p.window)) ? s[r] : kNegInf;
      }
      mx = fmaxf(mx, s[r]);
    }
    mx = xor32_max(mx);
    const bool up = mx > m_run + kMaxSlack;
    if (__builtin_amdgcn_ballot_w64(up)) {
      const float mn = up ? mx : m_run;
      const float alpha = up ? (m_run == kNegInf ? 0.f : __builtin_amdgcn_exp2f(m_run - mn)) : 1.f;
      m_run = mn;
      l_part *= alpha;
#pragma unroll
      for (int md = 0; md < MD; ++md) o[md] *= alpha;
    }
    const float mu = m_run == kNegInf ? 0.f : m_run;
    u32x4 pp[2][3];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float a = __builtin_amdgcn_exp2f(s[2 * i] - mu);
      const float b = __builtin_amdgcn_exp2f(s[2 * i + 1] - mu);
      l_part += a + b;
      unsigned x, y, z;
      split3(a, b, x, y, z);
      pp[i >> 2][0][i & 3] = x;
      pp[i >> 2][1][i & 3] = y;
      pp[i >> 2][2][i & 3] = z;
    }
    // ---- the next tile's loads, then O^T += V^T P^T over them ----
    const bool more = t < t_last;
    if (more) {
      fetch(t + 1, phys, kr, vr);
      phys = lookup(t + 2);
    }
#pragma unroll
    for (int j2 = 0; j2 < 2; ++j2)
#pragma unroll
      for (int md = 0; md < MD; ++md) {
        u32x4 va[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const char *src = s_v(buf) + j * VPART + (j2 * MD + md) * 1024 + 8 * lane;
          const u32x2 lo = lds_tr(src), hi = lds_tr(src + 512);
          va[j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
        }
        o[md] = mfma_x3(va, pp[j2], o[md]);
      }
    if (more) stage(buf ^ 1, kr, vr);
    __syncthreads();
  }

  const float l = xor32_sum(l_part);
  if (nsplit > 1) {
    // one split of the item, as in prefill_pipe_kernel (same layout)
    if (it.split == 0) {
      if (tid == 0) p.flags[(long)it.grp * p.max_tiles + it.qt] = odd != 0;
      if (it.qt == 0)
        for (int t = (it.len + rows - 1) / rows + tid; t < p.max_tiles; t += NT)
          p.flags[(long)it.grp * p.max_tiles + t] = 0;
    }
    const long unit = ((long)it.grp * p.max_tiles + it.qt) * p.max_splits + it.split;
    float *part = p.part + unit * prefill_part_floats(COLS, D) + (long)w * prefill_part_floats(32, D);
#pragma unroll
    for (int md = 0; md < MD; ++md)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        ((f32x4 *)part)[(md * 4 + q) * 64 + lane] =
            f32x4{o[md][4 * q], o[md][4 * q + 1], o[md][4 * q + 2], o[md][4 * q + 3]};
    part += 1024 * MD;
    if (h2 == 0) {
      part[l32] = m_run;
      part[32 + l32] = l;
    }
    return;
  }
  // ---- flag a result that the parts may not have held; normalise and store ----
  unsigned mb = 0;   // largest |O| of the column (as bits: infinities and NaNs compare above every finite value)
#pragma unroll
  for (int md = 0; md < MD; ++md)
#pragma unroll
    for (int r = 0; r < 16; ++r) mb = max(mb, __float_as_uint(o[md][r]) & 0x7fffffffu);
  mb = max(mb, (unsigned)__shfl_xor((int)mb, 32));
  const float top = __uint_as_float(mb) / l;
  const bool redo = odd || (colok && !(top >= kX3Least && top <= 3.0e38f));
  if (__builtin_amdgcn_ballot_w64(redo) && lane == 0) s_flag = 1;
  __syncthreads();
  if (tid == 0) p.flags[(long)it.grp * p.max_tiles + it.qt] = s_flag;
  if (it.qt == 0)
    for (int t = (it.len + rows - 1) / rows + tid; t < p.max_tiles; t += NT)
      p.flags[(long)it.grp * p.max_tiles + t] = 0;
  if (s_flag && prefill_redo_fits(G)) {
    prefill_redo<DD_F32, D, kX3Waves>(p, s_mem, it.grp, r0, r0 + rows_here);
    return;
  }
  if (!colok) return;
  const float inv = 1.f / l;
#pragma unroll
  for (int md = 0; md < MD; ++md)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int d = 32 * md + 8 * q + 4 * h2;
      if (D % 32 && d >= D) continue;
      *(f32x4 *)((float *)p.out + qrow + d) =
          f32x4{o[md][4 * q], o[md][4 * q + 1], o[md][4 * q + 2], o[md][4 * q + 3]} * inv;
    }
#endif  // __HIP_DEVICE_COMPILE__
}

template <int D>
int launch_x3(PrefillParams p, int max_len, hipStream_t s) {
  constexpr int COLS = 32 * kX3Waves;
  p.max_tiles = (int)dd_cdiv(max_len, COLS / p.G);
  const long items = (long)p.n * p.KH * p.max_tiles;
  if (p.max_splits <= 1) p.max_splits = 1, p.split_tiles = INT_MAX;
  const long grid = items * p.max_splits;
  if (grid == 0) return DD_OK;
  if (grid > 0x7fffffffL) return DD_EUNSUPPORTED;
  hipLaunchKernelGGL((prefill_x3_kernel<D>), dim3((unsigned)grid), dim3(64 * kX3Waves), 0, s, p);
  DD_LAUNCH_CHECK();
  if (p.max_splits > 1) {
    hipLaunchKernelGGL((prefill_merge_kernel<DD_F32, kX3Waves, kX3Keys, D>), dim3((unsigned)items, kX3Waves),
                       dim3(64 * ((D + 31) / 32)), 0, s, p);
    DD_LAUNCH_CHECK();
  }
  return DD_OK;
}

}  // namespace

int prefill_x3_dispatch(const PrefillParams &p, int dim, int max_len, hipStream_t s) {
  switch (dim) {
    case 16: return launch_x3<16>(p, max_len, s);
    case 32: return launch_x3<32>(p, max_len, s);
    case 48: return launch_x3<48>(p, max_len, s);
    case 64: return launch_x3<64>(p, max_len, s);
    case 80: return launch_x3<80>(p, max_len, s);
    case 96: return launch_x3<96>(p, max_len, s);
    case 112: return launch_x3<112>(p, max_len, s);
    case 128: return launch_x3<128>(p, max_len, s);
    default: return DD_EUNSUPPORTED;
  }
}

}  // namespace dd_prefill
