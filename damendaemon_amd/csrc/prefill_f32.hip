// Chunked-prefill attention in fp32 arithmetic on the matrix cores (gfx950):
// fp32 pages at any head size that is a multiple of 16 up to 256, and
// bf16 / fp16 pages at the head sizes the 16-bit MFMA kernels are not built
// for (e.g. 80, 96, 160).
//
// Same semantics as the other prefill kernels (damendaemon/paged.py:97-111
// with qwen2.py:754-770; fp32 pages are the fp32 compute_dtype of
// qwen2.py:403-409, and SDPA accepts any head size): query row j of segment
// i attends keys 0 .. start_i + j of its slot, and only keys > position -
// window when a window is set; GQA head h reads KV head h / G;
// softmax(q.k * scale) . v.
//
// Every product is exact fp32: Q, K and V (16-bit values widened exactly
// when they are loaded) and the probabilities enter v_mfma_f32_16x16x4_f32
// unrounded, accumulation is fp32; 16-bit outputs are rounded once at the
// end.
//
// Layout.  A workgroup of W = 8 waves (two per SIMD; at most 204 VGPRs up to
// D = 256) owns one (segment, KV head) and 16 W (query row, head) columns, a
// wave 16 of them with its Q in registers (lane (kg, n16): column n16, dims
// (D/4) kg ..+D/4).  Per step the workgroup stages a 32-key tile of K and V
// in LDS as fp32 (plain loads of the next tile are in flight while the
// current one is computed; double buffer, one barrier per step).  A wave
// forms S^T = K Q^T for its columns (16-key MFMA tiles, one MFMA per dim of
// the four each lane holds per 16-byte piece), the online softmax per column
// across the four lanes that hold it, and O^T += V^T P^T with key 4 kg + e of
// a 16-key tile as k-index kg of the e-th MFMA, so P^T is the softmax
// registers themselves.  O^T tile md row m holds dim (D/16) m + md, so a lane
// reads the D/16 contiguous dims of a V row.  LDS rows are padded by 16 bytes,
// so the 16-row K operand reads hit distinct banks.  Keys past the context or
// behind an unallocated page-table entry are staged as zeros (a zero
// probability then never meets a NaN).
#include "prefill_f32_item.h"

#include <climits>

namespace {

template <int DT, int D, int W>
__global__ __launch_bounds__(64 * W) void prefill_f32_kernel(PrefillGenericArgs p) {
#if __HIP_DEVICE_COMPILE__
  __shared__ __align__(16) char s_kv[f32_lds<D>()];
  const int G = p.heads / p.kv_heads;
  const int rows = 16 * W / G;
  if (!p.flags) {
    // one work item per workgroup, later query tiles (more keys) first
    const int ngrp = p.n * p.kv_heads;
    f32_item<DT, D, W>(p, s_kv, (int)(blockIdx.x % ngrp), rows * (p.max_tiles - 1 - (int)(blockIdx.x / ngrp)), INT_MAX);
    return;
  }
  // Re-run of the 16-bit kernel's flagged work items: workgroup b owns group
  // b and recomputes those of its query tiles that a flagged item covers.
  // Every flag of the group is defined (the 16-bit kernel zeroes those of
  // tiles past the segment), so the common case -- nothing flagged -- costs
  // one load per lane and no other memory access.
  const int grp = blockIdx.x;
  const int lane = threadIdx.x & 63;
  for (int f0 = 0; f0 < p.flag_tiles; f0 += 64) {
    const int f = f0 + lane;
    const unsigned long long hot =
        __builtin_amdgcn_ballot_w64(f < p.flag_tiles && p.flags[(long)grp * p.flag_tiles + f] != 0);
    if (!hot) continue;
    // query tiles of this kernel that overlap the flagged items f0 + bit
    for (int qt = (f0 * p.flag_rows) / rows; qt < p.max_tiles && qt * rows < (f0 + 64) * p.flag_rows; ++qt) {
      const int lo = qt * rows / p.flag_rows - f0, hi = ((qt + 1) * rows - 1) / p.flag_rows - f0;
      bool any = false;
      for (int b = lo < 0 ? 0 : lo; b <= hi && b < 64; ++b) any |= (hot >> b) & 1;
      if (!any) continue;
      __syncthreads();   // the previous item's LDS reads are done
      f32_item<DT, D, W>(p, s_kv, grp, qt * rows, INT_MAX);
    }
  }
#endif  // __HIP_DEVICE_COMPILE__
}

template <int DT, int D>
int launch_f32(PrefillGenericArgs a, hipStream_t s) {
  constexpr int W = 8;
  const int G = a.heads / a.kv_heads;
  if (G > 16 * W) return DD_EUNSUPPORTED;
  const int rows = 16 * W / G;
  a.max_tiles = (int)dd_cdiv(a.max_len, rows);
  const long grid = a.flags ? (long)a.n * a.kv_heads : (long)a.max_tiles * a.n * a.kv_heads;
  if (grid == 0) return DD_OK;
  if (grid > 0x7fffffffL) return DD_EUNSUPPORTED;
  hipLaunchKernelGGL((prefill_f32_kernel<DT, D, W>), dim3((unsigned)grid), dim3(64 * W), 0, s, a);
  DD_LAUNCH_CHECK();
  return DD_OK;
}

template <int DT>
int dispatch_f32(const PrefillGenericArgs &a, hipStream_t s) {
  switch (a.dim) {
    case 16: return launch_f32<DT, 16>(a, s);
    case 32: return launch_f32<DT, 32>(a, s);
    case 48: return launch_f32<DT, 48>(a, s);
    case 64: return launch_f32<DT, 64>(a, s);
    case 80: return launch_f32<DT, 80>(a, s);
    case 96: return launch_f32<DT, 96>(a, s);
    case 112: return launch_f32<DT, 112>(a, s);
    case 128: return launch_f32<DT, 128>(a, s);
    case 160: return launch_f32<DT, 160>(a, s);
    case 176: return launch_f32<DT, 176>(a, s);
    case 192: return launch_f32<DT, 192>(a, s);
    case 208: return launch_f32<DT, 208>(a, s);
    case 224: return launch_f32<DT, 224>(a, s);
    case 240: return launch_f32<DT, 240>(a, s);
    case 256: return launch_f32<DT, 256>(a, s);
    default: return DD_EUNSUPPORTED;
  }
}

}  // namespace

int dd_prefill_f32(const PrefillGenericArgs &a, int dtype, hipStream_t s) {
  if (a.kv_heads <= 0 || a.heads % a.kv_heads) return DD_EUNSUPPORTED;
  if (dtype == DD_F32) return dispatch_f32<DD_F32>(a, s);
  if (dtype == DD_BF16) return dispatch_f32<DD_BF16>(a, s);
  if (dtype == DD_F16) return dispatch_f32<DD_F16>(a, s);
  return DD_EUNSUPPORTED;
}
