// Device pieces shared by the GEMM kernels (gemm.hip, gemm_ring.hip): the
// workgroup -> tile mapping, the LDS chunk swizzle and the epilogue of four
// consecutive output columns.
#pragma once

#include "common.hpp"
#include "tx_internal.hpp"

namespace tx {

// Workgroup -> tile mapping.  Workgroups are dispatched round-robin over the
// 8 XCDs (workgroup i runs on XCD i % 8); remap so that each XCD receives a
// contiguous range of logical tiles, then walk tiles in groups of GROUP tile
// rows so that concurrently running tiles share A rows and W columns in L2.
__device__ __forceinline__ void gemm_tile_of(int pid, int nwg, int tiles_m, int tiles_n,
                                             int& tm, int& tn, int GROUP = 8) {
  const int x = pid & 7, i = pid >> 3, q = nwg >> 3, r = nwg & 7;
  pid = x * q + (x < r ? x : r) + i;
  const int width = GROUP * tiles_n;
  const int group = pid / width;
  const int first_m = group * GROUP;
  const int gsz = (tiles_m - first_m) < GROUP ? (tiles_m - first_m) : GROUP;
  const int in_group = pid - group * width;
  tm = first_m + in_group % gsz;
  tn = in_group / gsz;
}

template <int CH>
__device__ __forceinline__ int big_swz(int r) {
  // CH = 16-byte chunks per LDS row.  16 consecutive rows read at one
  // logical chunk must cover all 64 banks.  A ds_read_b128 serves 16 lanes
  // per cycle from 64 four-byte banks, and the bank group of a 16-byte unit
  // (measured with SQ_LDS_BANK_CONFLICT on gfx950 over seven access
  // patterns) is address bits 4..7 with bit 10 folded into bit 4: with
  // 128-byte rows, rows r and r + 8 already differ in that bit, so the row's
  // low three bits are the whole swizzle.  Also folding in bit 3 of the row
  // cancels the hardware's term and pairs rows r and r + 8 (two cycles per
  // read instead of one).
  if constexpr (CH == 8) return r & 7;
  else return (r >> 2) & 3;
}

// ------------------------------------------------------ shared epilogue
// Epilogue of four consecutive output columns n..n+3 of row m (the D^T
// accumulator layout: lane holds columns, not rows).  acc: the fp32 sums;
// bv: the bias values (0 without BIAS); rv: the residual values (read before
// any store of the group, since the residual may alias C); valid: the row's
// row_valid flag (true without masks).
__device__ __forceinline__ bool gemm_row_valid(const GemmArgs& g, int m) {
  const bool need = (g.epi & (TX_EPI_MASK_DELTA | TX_EPI_MASK_OUT)) && g.row_valid != nullptr;
  return !need || g.row_valid[m] != 0;
}
template <typename TC, bool QKV>
__device__ __forceinline__ void gemm_finish4(const GemmArgs& g, int m, int n, const float* acc,
                                             const float* bv, const float* rv, bool valid) {
  const uint32_t epi = g.epi;
  TC* __restrict__ C = (TC*)g.c;
  if (!QKV && (epi & TX_EPI_SPLIT_OUT)) {
    // fp32-residual policy: the unrounded value as a hi/lo pair.
    float hi[4], lo[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float t = acc[e] + bv[e];
      if (epi & TX_EPI_GELU_ERF) t = gelu_erf(t);
      hi[e] = round_to<TC>(t);
      lo[e] = t - hi[e];
    }
    store4<TC>(C + (int64_t)m * g.ldc + n, hi);
    store4<TC>(C + (int64_t)m * g.ldc + n + g.n, lo);
    return;
  }
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float t = round_to<TC>(acc[e] + bv[e]);
    if (epi & TX_EPI_GELU_ERF) t = round_to<TC>(gelu_erf(t));
    v[e] = t;
  }
  if (!QKV) {
    if (epi & TX_EPI_RESIDUAL) {
      const bool drop = (epi & TX_EPI_MASK_DELTA) && !valid;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = round_to<TC>(rv[e] + (drop ? 0.f : v[e]));
    }
    if ((epi & TX_EPI_MASK_OUT) && !valid) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = 0.f;
    }
  }
  if (!QKV || n < g.qk_cols) {
    store4<TC>(C + (int64_t)m * g.ldc + n, v);
  } else {
    // V columns go head-transposed into vt[b][h][d][s].
    const int nv = n - g.qk_cols;
    const int hh = nv / g.head_dim, d0 = nv - hh * g.head_dim;
    const int b = m / g.seq, sq = m - b * g.seq;
    TC* dst = (TC*)g.vt + ((int64_t)(b * g.heads + hh) * g.head_dim + d0) * g.ldvt + sq;
#pragma unroll
    for (int e = 0; e < 4; ++e) dst[(int64_t)e * g.ldvt] = from_f32<TC>(v[e]);
  }
}

}  // namespace tx
