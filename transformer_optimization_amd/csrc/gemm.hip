// bf16/fp16 GEMM on gfx950 MFMA (v_mfma_f32_32x32x16_*) with fused epilogues.
//
//   C[m, n] = epilogue( sum_k A[m, k] * W[n, k] )
//
// A is the activation [M, K] (row-major), W is nn.Linear storage [N, K]
// (row-major), so both operands are K-contiguous and every MFMA operand is a
// single 128-bit LDS read.  Replaces F.linear / _triton_linear /
// _triton_gemm_gelu on the hot path (TTB:1754-1803, 1860-1880).
//
// Structure: a workgroup computes a BM x BN tile with WM x WN waves, each
// wave a (BM/WM) x (BN/WN) sub-tile of 32x32 MFMA blocks.  K advances in
// steps of 64; the next K step is fetched from HBM into registers while the
// current one is multiplied out of LDS (two LDS stages, one barrier per
// step).  LDS rows are 128 bytes (64 x 16-bit); the 16-byte chunk c of row r
// is stored at chunk c ^ swz(r) so that both the cooperative row writes and
// the MFMA fragment reads (16 rows x one chunk) touch distinct banks.
//
// Epilogue (rounding points of the eager chain, TTB:1795-1798, 4311-4312):
//   v = round_C(acc + bias)          BIAS
//   v = round_C(gelu_erf(v))         GELU_ERF  (reads the rounded value)
//   v = round_C(residual + v)        RESIDUAL  (x + sublayer(x))
// with row masks for padded tokens.  The packed-QKV variant writes columns
// [0, 2D) to qk[M, 2D] and the V columns head-transposed into vt.
#include <cstdlib>

#include "common.hpp"
#include "gemm_common.hpp"
#include "gemm_route.hpp"
#include "tx_internal.hpp"

namespace tx {

constexpr int GEMM_BK = 64;

// LDS chunk swizzle: bijective on rows 0..7 and 8..15, and on the even and
// the odd rows of any 16-row group, so 8-lane (128 B) and 16-lane (256 B)
// access phases are both conflict-free.
__device__ __forceinline__ int gemm_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

template <typename T, typename TC, typename TB, typename TR, int BM, int BN, int WM, int WN, bool QKV>
__global__ __launch_bounds__(WM* WN * 64) void gemm_kernel(GemmArgs g) {
  constexpr int NT = WM * WN * 64;
  constexpr int BK = GEMM_BK;
  constexpr int TM = BM / WM, TN = BN / WN;
  constexpr int FM = TM / 32, FN = TN / 32;
  constexpr int A_CH = BM * 8 / NT, B_CH = BN * 8 / NT;  // 16-byte chunks per thread
  static_assert(A_CH * NT == BM * 8 && B_CH * NT == BN * 8, "tile/thread mismatch");
  static_assert(FM >= 1 && FN >= 1, "wave tile too small");
  typedef typename Mfma<T>::vec vec;

  __shared__ __attribute__((aligned(16))) T lds[2][(BM + BN) * BK];

  const int tiles_m = (g.m + BM - 1) / BM, tiles_n = (g.n + BN - 1) / BN;
  int tm, tn;
  gemm_tile_of(blockIdx.x, gridDim.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const T* __restrict__ A = (const T*)g.a;
  const T* __restrict__ W = (const T*)g.w;

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  u32x4 ra[A_CH], rb[B_CH];
  const int KT = (g.k + BK - 1) / BK;

  auto gload = [&](int kt) {
    const int k0 = kt * BK;
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      const int idx = tid + i * NT, row = idx >> 3, cc = idx & 7;
      const int gm = m0 + row, gk = k0 + cc * 8;
      if (gm < g.m && gk < g.k) {
        ra[i] = ld128(A + (int64_t)gm * g.lda + gk);
      } else {
        ra[i] = u32x4{0u, 0u, 0u, 0u};
      }
    }
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
      const int idx = tid + i * NT, row = idx >> 3, cc = idx & 7;
      const int gn = n0 + row, gk = k0 + cc * 8;
      if (gn < g.n && gk < g.k) {
        rb[i] = ld128(W + (int64_t)gn * g.ldw + gk);
      } else {
        rb[i] = u32x4{0u, 0u, 0u, 0u};
      }
    }
  };
  auto lstore = [&](int stage) {
    T* As = lds[stage];
    T* Bs = lds[stage] + BM * BK;
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      const int idx = tid + i * NT, row = idx >> 3, cc = idx & 7;
      st128(As + row * BK + ((cc ^ gemm_swz(row)) << 3), ra[i]);
    }
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
      const int idx = tid + i * NT, row = idx >> 3, cc = idx & 7;
      st128(Bs + row * BK + ((cc ^ gemm_swz(row)) << 3), rb[i]);
    }
  };

  const int frag_r = lane & 31;       // row within a 32-row MFMA block
  const int frag_h = lane >> 5;       // which 8-wide k half of a 16-wide k step
  const int a_row0 = wm * TM, b_row0 = wn * TN;

  gload(0);
  lstore(0);
  __syncthreads();
  for (int kt = 0; kt < KT; ++kt) {
    const int st = kt & 1;
    if (kt + 1 < KT) gload(kt + 1);
    const T* As = lds[st];
    const T* Bs = lds[st] + BM * BK;
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      const int ch = 2 * ks + frag_h;
      vec af[FM], bf[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int r = a_row0 + 32 * i + frag_r;
        af[i] = *reinterpret_cast<const vec*>(As + r * BK + ((ch ^ gemm_swz(r)) << 3));
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int r = b_row0 + 32 * j + frag_r;
        bf[j] = *reinterpret_cast<const vec*>(Bs + r * BK + ((ch ^ gemm_swz(r)) << 3));
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = Mfma<T>::mma32(af[i], bf[j], acc[i][j]);
    }
    if (kt + 1 < KT) lstore(st ^ 1);
    __syncthreads();
  }

  // ---------------------------------------------------------------- epilogue
  const uint32_t epi = g.epi;
  const TB* __restrict__ bias = (const TB*)g.bias;
  const TR* __restrict__ res = (const TR*)g.res;
  TC* __restrict__ C = (TC*)g.c;
  const bool need_valid = (epi & (TX_EPI_MASK_DELTA | TX_EPI_MASK_OUT)) && g.row_valid != nullptr;
  const bool split = !QKV && (epi & TX_EPI_SPLIT_OUT);

#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int col = n0 + b_row0 + 32 * j + (lane & 31);
    if (col >= g.n) continue;
    const float bval = (epi & TX_EPI_BIAS) ? to_f32(bias[col]) : 0.f;
    const bool to_vt = QKV && col >= g.qk_cols;
    int vt_h = 0, vt_d = 0;
    if (QKV && to_vt) {
      const int nv = col - g.qk_cols;
      vt_h = nv / g.head_dim;
      vt_d = nv - vt_h * g.head_dim;
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int row0 = m0 + a_row0 + 32 * i + 8 * q4 + 4 * (lane >> 5);
        if (split) {
          // fp32-residual policy: the exact fp32 value as a hi/lo pair.
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = row0 + e;
            float t = acc[i][j][4 * q4 + e] + bval;
            if (epi & TX_EPI_GELU_ERF) t = gelu_erf(t);
            const TC hi = from_f32<TC>(t);
            const TC lo = from_f32<TC>(t - to_f32(hi));
            if (row < g.m) {
              C[(int64_t)row * g.ldc + col] = hi;
              C[(int64_t)row * g.ldc + col + g.n] = lo;
            }
          }
          continue;
        }
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = row0 + e;
          float t = round_to<TC>(acc[i][j][4 * q4 + e] + bval);
          if (epi & TX_EPI_GELU_ERF) t = round_to<TC>(gelu_erf(t));
          if (!QKV && row < g.m) {
            const bool valid = !need_valid || g.row_valid[row] != 0;
            if (epi & TX_EPI_RESIDUAL) {
              const float dlt = ((epi & TX_EPI_MASK_DELTA) && !valid) ? 0.f : t;
              t = round_to<TC>(to_f32(res[(int64_t)row * g.ldr + col]) + dlt);
            }
            if ((epi & TX_EPI_MASK_OUT) && !valid) t = 0.f;
          }
          v[e] = t;
        }
        if (!to_vt) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (row0 + e < g.m) C[(int64_t)(row0 + e) * g.ldc + col] = from_f32<TC>(v[e]);
        } else if constexpr (QKV && sizeof(TC) == 2) {
          // V^T store: consecutive rows are consecutive sequence positions.
          const int b = row0 / g.seq, s = row0 - b * g.seq;
          TC* dst = (TC*)g.vt + ((int64_t)(b * g.heads + vt_h) * g.head_dim + vt_d) * g.ldvt;
          if ((g.seq & 3) == 0 && row0 + 3 < g.m) {
            u32x2 pk;
            pk[0] = pack2<TC>(v[0], v[1]);
            pk[1] = pack2<TC>(v[2], v[3]);
            st64(dst + s, pk);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int row = row0 + e;
              if (row < g.m) {
                const int bb = row / g.seq, ss = row - bb * g.seq;
                TC* d2 = (TC*)g.vt + ((int64_t)(bb * g.heads + vt_h) * g.head_dim + vt_d) * g.ldvt;
                d2[ss] = from_f32<TC>(v[e]);
              }
            }
          }
        }
      }
    }
  }
}

// ================================================================ big tiles
// gemm_big_kernel: 128 x 128 / 256 x 256 tiles, compiler-scheduled; the
// baseline gemm_hp_kernel is measured against (variants 20 / 19).
//
// Persistent: the grid holds at most as many workgroups as fit on the CUs
// at once (LDS-bound: one for the default tiles) and workgroup w
// computes tiles w, w + G, w + 2G, ... (G = grid size), each mapped through
// gemm_tile_of.  A BM x BN x BK block of both operands moves from global
// memory straight into LDS (global_load_lds_dwordx4: each lane's 16 bytes
// land at lds + 16 * lane, so the XOR swizzle is applied by choosing which
// global chunk each lane fetches).  STAGES LDS buffers form one ring over the
// workgroup's whole sequence of (tile, k step) pairs: at step s the waves
// wait for stage s, refill the stage read at step s - 1 with step
// s + STAGES - 1 -- which belongs to the next tile near the end of a tile --
// and multiply stage s.  The next tile's first operands are therefore in
// flight while the current tile's epilogue runs, and global latency is
// covered by STAGES - 1 steps of MFMA work.
//
// The product is formed transposed, D^T = W A^T (W rows are the MFMA A
// operand): lane l then holds four consecutive output columns of one output
// row, so the epilogue reads bias / residual and writes C in 8-byte (16-bit
// C) or 16-byte (fp32 C) vectors.  Per output element the MFMA sequence is
// the same as in gemm_kernel (k ascending in steps of 16), so both kernels
// produce identical bits.
//
// OPT bit 0: raise the wave priority around each MFMA group; bit 1: issue
// the next stage's loads after the first k16 group instead of right after
// the barrier (the fragment reads of that group then go out first); bit 2:
// read the fragments of the next k16 group while the MFMAs of this one run.
// The defaults use bits 1 and 2 (the priority raise is a scheduling fence
// that keeps the compiler from hoisting the fragment reads).
// Workgroups of one tile shape resident per CU, bounded by its LDS ring
// (160 KB per CU); the register budget (the launch bound's minimum waves per
// SIMD) is sized to keep that many resident.
template <typename T, int BM, int BN, int BK, int STAGES>
constexpr int big_per_cu() {
  return (160 * 1024) / (STAGES * (BM + BN) * BK * (int)sizeof(T));
}
template <typename T, int BM, int BN, int BK, int STAGES, int NW>
constexpr int big_waves_per_simd() {
  const int w = big_per_cu<T, BM, BN, BK, STAGES>() * NW / 4;
  return w < 1 ? 1 : (w > 4 ? 4 : w);
}

template <typename T, typename TC, typename TB, typename TR, int BM, int BN, int BK, int WM, int WN,
          int STAGES, int OPT, bool QKV>
__global__ __launch_bounds__(WM* WN * 64, (big_waves_per_simd<T, BM, BN, BK, STAGES, WM * WN>()))
void gemm_big_kernel(GemmArgs g) {
  constexpr int NW = WM * WN;
  constexpr int CH = BK / 8;                 // 16-byte chunks per LDS row
  constexpr int RPI = 64 / CH;               // LDS rows filled by one wave instruction
  constexpr int A_LD = BM / RPI / NW;        // wave instructions per stage for A
  constexpr int B_LD = BN / RPI / NW;
  constexpr int LPW = A_LD + B_LD;
  constexpr int TM = BM / WM, TN = BN / WN;
  constexpr int FM = TM / 32, FN = TN / 32;
  constexpr int KS = BK / 16;
  static_assert(A_LD * RPI * NW == BM && B_LD * RPI * NW == BN, "load split");
  static_assert(FM >= 1 && FN >= 1, "wave tile");
  typedef typename Mfma<T>::vec vec;

  __shared__ __attribute__((aligned(16))) T lds[STAGES][(BM + BN) * BK];

  const int tiles_m = (g.m + BM - 1) / BM, tiles_n = (g.n + BN - 1) / BN;
  const int n_tiles = tiles_m * tiles_n;
  const int my_tiles = (n_tiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  const int KT = g.k / BK;
  const int total = my_tiles * KT;  // steps of this workgroup
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  // ---- loader state: the tile / k step of the most recent issue.
  const T* __restrict__ A = (const T*)g.a;
  const T* __restrict__ W = (const T*)g.w;
  const int lr = lane / CH, lp = lane % CH;
  const T* asrc[A_LD];
  const T* bsrc[B_LD];
  int ld_ti = -1, ld_kt = KT - 1;
  auto point_at = [&](int ti) {
    int tm, tn;
    gemm_tile_of((int)blockIdx.x + ti * (int)gridDim.x, n_tiles, tiles_m, tiles_n, tm, tn, g.group);
#pragma unroll
    for (int i = 0; i < A_LD; ++i) {
      const int row = (i * NW + wave) * RPI + lr;
      const int gm = min(tm * BM + row, g.m - 1);  // rows past M feed discarded outputs
      asrc[i] = A + (int64_t)gm * g.lda + 8 * (lp ^ big_swz<CH>(row));
    }
#pragma unroll
    for (int i = 0; i < B_LD; ++i) {
      const int row = (i * NW + wave) * RPI + lr;
      const int gn = min(tn * BN + row, g.n - 1);
      bsrc[i] = W + (int64_t)gn * g.ldw + 8 * (lp ^ big_swz<CH>(row));
    }
  };
  // Issue global step `s` (steps past the end repeat the last one into a
  // stage that is never read, so every step issues LPW loads per wave).
  auto issue = [&](int s) {
    if (s < total) {
      if (++ld_kt == KT) {
        ld_kt = 0;
        point_at(++ld_ti);
      }
    }
    const int k0 = ld_kt * BK;
    T* As = lds[s % STAGES];
    T* Bs = As + BM * BK;
#pragma unroll
    for (int i = 0; i < A_LD; ++i)
      dma16(asrc[i] + k0, As + (i * NW + wave) * RPI * BK);
#pragma unroll
    for (int i = 0; i < B_LD; ++i)
      dma16(bsrc[i] + k0, Bs + (i * NW + wave) * RPI * BK);
  };

  const int wm = wave / WN, wn = wave % WN;
  const int fr = lane & 31, half = lane >> 5;
  const int fs = big_swz<CH>(fr);  // row swizzle of every fragment row of this lane
  int koff[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koff[ks] = 8 * ((2 * ks + half) ^ fs);
  const int a_row = (wm * TM + fr) * BK, b_row = (wn * TN + fr) * BK;

  const uint32_t epi = g.epi;
  const TB* __restrict__ bias = (const TB*)g.bias;
  const TR* __restrict__ res = (const TR*)g.res;

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) issue(s);

  for (int ti = 0; ti < my_tiles; ++ti) {
    int tm, tn;
    gemm_tile_of((int)blockIdx.x + ti * (int)gridDim.x, n_tiles, tiles_m, tiles_n, tm, tn, g.group);
    const int m0 = tm * BM, n0 = tn * BN;

    f32x16 acc[FN][FM];
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.f;

    for (int kt = 0; kt < KT; ++kt) {
      const int s = ti * KT + kt;
      // Wait for this wave's share of stage s, then for every wave's.
      ring_barrier<LPW * (STAGES - 2)>();
      if (!(OPT & 2)) issue(s + STAGES - 1);
      const T* As = lds[s % STAGES] + a_row;
      const T* Bs = lds[s % STAGES] + BM * BK + b_row;
      if constexpr (OPT & 4) {
        // The fragments of k step ks + 1 are read while the MFMAs of ks run
        // (two fragment buffers): one LDS latency per stage instead of one
        // per k step.
        vec af[2][FM], bf[2][FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) af[0][i] = *reinterpret_cast<const vec*>(As + 32 * i * BK + koff[0]);
#pragma unroll
        for (int j = 0; j < FN; ++j) bf[0][j] = *reinterpret_cast<const vec*>(Bs + 32 * j * BK + koff[0]);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int cb = ks & 1, nb = cb ^ 1;
          if (ks + 1 < KS) {
#pragma unroll
            for (int i = 0; i < FM; ++i) af[nb][i] = *reinterpret_cast<const vec*>(As + 32 * i * BK + koff[ks + 1]);
#pragma unroll
            for (int j = 0; j < FN; ++j) bf[nb][j] = *reinterpret_cast<const vec*>(Bs + 32 * j * BK + koff[ks + 1]);
          }
          if (OPT & 1) __builtin_amdgcn_s_setprio(1);
#pragma unroll
          for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int i = 0; i < FM; ++i) acc[j][i] = Mfma<T>::mma32(bf[cb][j], af[cb][i], acc[j][i]);
          if (OPT & 1) __builtin_amdgcn_s_setprio(0);
          if ((OPT & 2) && ks == 0) issue(s + STAGES - 1);
        }
      } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          vec af[FM], bf[FN];
#pragma unroll
          for (int i = 0; i < FM; ++i) af[i] = *reinterpret_cast<const vec*>(As + 32 * i * BK + koff[ks]);
#pragma unroll
          for (int j = 0; j < FN; ++j) bf[j] = *reinterpret_cast<const vec*>(Bs + 32 * j * BK + koff[ks]);
          if (OPT & 1) __builtin_amdgcn_s_setprio(1);
#pragma unroll
          for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int i = 0; i < FM; ++i) acc[j][i] = Mfma<T>::mma32(bf[j], af[i], acc[j][i]);
          if (OPT & 1) __builtin_amdgcn_s_setprio(0);
          if ((OPT & 2) && ks == 0) issue(s + STAGES - 1);
        }
      }
    }

    // -------------------------------------------------------------- epilogue
    // acc[j][i][4*q4 + e]: row m = m0 + wm*TM + 32i + fr,
    //                      col n = n0 + wn*TN + 32j + 8*q4 + 4*half + e.
    // The reads of a 32-column group (bias, residual rows, row flags) are all
    // issued before the first is used: one memory latency per group rather
    // than one per read.  Their addresses are clamped into the operands;
    // rows and columns past the edge are never stored.
    // Every read is consumed (settle) on every path before the next tile's K
    // loop: a read left pending there would make the compiler wait for it
    // (vmcnt) inside that loop, which also drains the DMA ring.
    int valid[FM];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if (j == 0) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
          valid[i] = QKV || gemm_row_valid(g, min(m0 + wm * TM + 32 * i + fr, g.m - 1));
      }
      typename Raw4<TB>::type braw[4];
      typename Raw4<TR>::type rraw[4][FM];
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int nc = min(n0 + wn * TN + 32 * j + 8 * q4 + 4 * half, g.n - 4);
        braw[q4] = {};
        if (epi & TX_EPI_BIAS) braw[q4] = ld_raw4(bias + nc);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          rraw[q4][i] = {};
          if (!QKV && (epi & TX_EPI_RESIDUAL)) {
            const int mc = min(m0 + wm * TM + 32 * i + fr, g.m - 1);
            rraw[q4][i] = ld_raw4(res + (int64_t)mc * g.ldr + nc);
          }
        }
      }
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        settle(braw[q4]);
#pragma unroll
        for (int i = 0; i < FM; ++i) settle(rraw[q4][i]);
      }
      if (j == 0) {
#pragma unroll
        for (int i = 0; i < FM; ++i) settle(valid[i]);
      }
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int n = n0 + wn * TN + 32 * j + 8 * q4 + 4 * half;
        if (n >= g.n) continue;
        float bv[4];
        unpack4<TB>(braw[q4], bv);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const int m = m0 + wm * TM + 32 * i + fr;
          if (m >= g.m) continue;
          float rv[4], a4[4];
          unpack4<TR>(rraw[q4][i], rv);
#pragma unroll
          for (int e = 0; e < 4; ++e) a4[e] = acc[j][i][4 * q4 + e];
          gemm_finish4<TC, QKV>(g, m, n, a4, bv, rv, valid[i] != 0);
        }
      }
    }
  }
  ring_drain();
}

// ================================================================ 256-row tiles
// gemm_hp_kernel: the main path for M >= 256 and K a multiple of 64.
//
// 256 x BN tiles (BN = 128, 192 or 256), eight waves as 2 x 4 (two per
// SIMD), each wave a 128 x BN/4 block of 16 x 16 output blocks
// (v_mfma_f32_16x16x32: FM x FN = 8 x BN/64 accumulators of four fp32), one
// workgroup per CU, persistent over tiles.  Against the 128 x 128 tiles of
// gemm_big_kernel this halves the operand bytes moved from L2 into LDS per
// FLOP, and the k32 MFMAs give the schedule twice as many issue slots to
// spread the fragment reads and DMA issues over.
//
// K advances in steps of 64 (two k32 groups) through NS LDS stages (two; three
// for 128-wide tiles, whose three stages fit in LDS) fed by
// global_load_lds_dwordx4.  The order of instructions inside a step is fixed
// by hand (every MFMA slot is closed by a scheduling barrier):
//   g0: the NQ MFMAs of group 0, with the fragment reads of group 1 spread
//       evenly between them;
//   barrier: this wave's DMA of step s + 1 has landed, every wave's too, and
//       every wave has read all of stage s % NS (group 1 was read during g0);
//   g1: the MFMAs of group 1, with the fragment reads of group 0 of step
//       s + 1 between them and the DMA issues of step s + NS (into the stage
//       the barrier released) in its first half.
// Fragment reads run one group ahead of their MFMAs; a DMA has at least half
// of g1 and all of the next g0 to land (issuing it early is what matters
// inside the forward, where weights come from HBM: 2-3% per forward against
// spreading it over all of g1).  The second wave on each SIMD covers what
// one wave leaves exposed (barrier skew, a memory instruction that cannot
// issue yet).  Steps run across tiles: the next tile's first steps load while
// the current tile's epilogue runs.
//
// Per output element the products are accumulated with k ascending, as in
// gemm_big_kernel and gemm_kernel; the three give identical bits (and equal
// F.linear bitwise at every c3/c4 shape).
template <typename T, typename TC, typename TB, typename TR, int BN, bool QKV, int NS = 2>
__global__ __launch_bounds__(512, 1) void gemm_hp_kernel(GemmArgs g) {
  constexpr int BM = 256, BK = 64, NW = 8, WNN = 4;
  static_assert(NS == 2 || NS == 3, "two or three K stages");
  constexpr int CH = BK / 8;     // 16-byte chunks per LDS row
  constexpr int RPI = 64 / CH;   // LDS rows filled by one DMA instruction
  constexpr int TM = BM / 2, TN = BN / WNN;
  constexpr int FM = TM / 16, FN = TN / 16;
  constexpr int A_LD = BM / RPI / NW, B_LD = BN / RPI / NW, LPW = A_LD + B_LD;
  constexpr int NR = FM + FN;    // fragment reads per group
  constexpr int NQ = FM * FN;    // MFMAs per group
  // A-major MFMA order (A fragments reloaded in place) for the 192-wide
  // tiles: without it that kernel spills 6-16 registers; with it, none, and
  // it runs 2-6% faster at the c3/c4 shapes.  The 256-wide kernel spills
  // either way, and is 25-35% slower in this order.
  constexpr bool AMAJ = BN == 192;
  constexpr int STAGE = (BM + BN) * BK;
  static_assert(B_LD * RPI * NW == BN && A_LD * RPI * NW == BM, "load split");
  static_assert(NR <= NQ && LPW <= NQ, "slots");
  typedef typename Mfma16<T>::vec vec;

  // LDS: the NS K stages, then one epilogue staging region per wave (16
  // output rows of TN 16-bit values, rows padded by 8 elements).
  constexpr int ES = TN + 8;
  __shared__ __attribute__((aligned(16))) T lds[NS * STAGE + NW * 16 * ES];

  const int tiles_m = (g.m + BM - 1) / BM, tiles_n = (g.n + BN - 1) / BN;
  const int n_tiles = tiles_m * tiles_n;
  const int my_tiles = (n_tiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  const int KT = g.k / BK;
  const int total = my_tiles * KT;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);

  // ---- loader: uniform tile bases, per-lane byte offsets (rows past the
  // edge are clamped into the operand; they feed discarded outputs).  Row
  // (i * NW + wave) * RPI + lr of a tile is the lane's row of issue i; its
  // low three bits are lr, so the chunk swizzle is a lane constant and a
  // clamped row keeps its own chunk.
  //   BN < 256: the offsets of every issue are formed once per tile and
  //   held in registers.
  //   BN = 256: that kernel has no registers to hold them (its accumulators
  //   take half of a wave's 256; held, they were spilled and reloaded beside
  //   the DMA issues, each reload waiting for every load in flight), so each
  //   issue forms its offset from a lane constant and the tile's uniform row
  //   limit, three vector ops.  (The same in the narrower kernels cost them
  //   2-6%.)
  static_assert(CH == 8 && RPI == 8, "eight 16-byte chunks per LDS row");
  constexpr bool LIVE_OFF = BN == 256;
  const int lr = lane / CH, lp = lane % CH;
  const uint32_t chk = (uint32_t)(8 * (lp ^ big_swz<CH>(lr)) * (int)sizeof(T));
  const uint32_t a_row0 = (uint32_t)((wave * RPI + lr) * (int)g.lda * (int)sizeof(T));
  const uint32_t b_row0 = (uint32_t)((wave * RPI + lr) * (int)g.ldw * (int)sizeof(T));
  const uint32_t a_step = (uint32_t)(NW * RPI * (int)g.lda * (int)sizeof(T));
  const uint32_t b_step = (uint32_t)(NW * RPI * (int)g.ldw * (int)sizeof(T));
  uint32_t a_lim = 0, b_lim = 0;  // byte offset of the tile's last valid row
  uint32_t aoff[LIVE_OFF ? 1 : A_LD], boff[LIVE_OFF ? 1 : B_LD];
  const char* abase = (const char*)g.a;
  const char* bbase = (const char*)g.w;
  int ld_ti = -1, ld_kt = KT - 1;
  auto point_at = [&](int ti) {
    int tm, tn;
    gemm_tile_of((int)blockIdx.x + ti * (int)gridDim.x, n_tiles, tiles_m, tiles_n, tm, tn, g.group);
    abase = (const char*)g.a + (int64_t)tm * BM * g.lda * (int64_t)sizeof(T);
    bbase = (const char*)g.w + (int64_t)tn * BN * g.ldw * (int64_t)sizeof(T);
    a_lim = (uint32_t)(min(g.m - 1 - tm * BM, BM - 1) * (int)g.lda * (int)sizeof(T));
    b_lim = (uint32_t)(min(g.n - 1 - tn * BN, BN - 1) * (int)g.ldw * (int)sizeof(T));
    if constexpr (!LIVE_OFF) {
#pragma unroll
      for (int i = 0; i < A_LD; ++i) aoff[i] = min(a_row0 + (uint32_t)i * a_step, a_lim) + chk;
#pragma unroll
      for (int i = 0; i < B_LD; ++i) boff[i] = min(b_row0 + (uint32_t)i * b_step, b_lim) + chk;
    }
  };
  // DMA issue q (0 .. LPW-1) of step s; q == 0 advances the loader to s
  // (steps past the end repeat the last one into a stage never read).
  const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)lds;
  auto dma = [&](int s, int q) {
    if (q == 0 && s < total) {
      if (++ld_kt == KT) {
        ld_kt = 0;
        point_at(++ld_ti);
      }
    }
    const int kb = ld_kt * BK * (int)sizeof(T);
    const uint32_t st = lds0 + (uint32_t)((s % NS) * STAGE * (int)sizeof(T));
    uint32_t off;
    if constexpr (LIVE_OFF) {
      // Formed at the issue: the opaque copy keeps the compiler from holding
      // one row offset per issue across the loop.
      uint32_t r0 = q < A_LD ? a_row0 : b_row0;
      asm volatile("" : "+v"(r0));
      off = q < A_LD ? min(r0 + (uint32_t)q * a_step, a_lim) + chk
                     : min(r0 + (uint32_t)(q - A_LD) * b_step, b_lim) + chk;
    } else {
      off = q < A_LD ? aoff[q] : boff[q - A_LD];
    }
    if (q < A_LD)
      dma16_m0(abase + kb, off, st + (uint32_t)((q * NW + wave) * RPI * BK * (int)sizeof(T)));
    else
      dma16_m0(bbase + kb, off, st + (uint32_t)((BM * BK + ((q - A_LD) * NW + wave) * RPI * BK) * (int)sizeof(T)));
  };

  // ---- fragment reads: read q (0 .. NR-1) of group grp of step s, in the
  // order the MFMAs consume them (W fragment 0, the FM A fragments, then W
  // fragments 1 .. FN-1).  Lane l supplies row l & 15 of a 16-row fragment,
  // the 8-wide k chunk l >> 4 of the group's 32.
  const int wm = wave / WNN, wn = wave % WNN;
  const int fr = lane & 15, kh = lane >> 4;
  const int fs = big_swz<CH>(fr);
  const int a_row = (wm * TM + fr) * BK, b_row = BM * BK + (wn * TN + fr) * BK;
  vec fa[2][FM], fb[2][FN];
  auto frag = [&](int s, int grp, int q, vec* a, vec* b) {
    const T* base = lds + (s % NS) * STAGE + 8 * ((4 * grp + kh) ^ fs);
    if (q == 0) b[0] = *reinterpret_cast<const vec*>(base + b_row);
    else if (q <= FM) a[q - 1] = *reinterpret_cast<const vec*>(base + a_row + 16 * (q - 1) * BK);
    else b[q - FM] = *reinterpret_cast<const vec*>(base + b_row + 16 * (q - FM) * BK);
  };

  const uint32_t epi = g.epi;
  const TB* __restrict__ bias = (const TB*)g.bias;
  const TR* __restrict__ res = (const TR*)g.res;

  // ---- prologue: steps 0 .. NS-1 in flight, group 0 of step 0 read.
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int q = 0; q < LPW; ++q) dma(s, q);
  ring_barrier<LPW * (NS - 1)>();
#pragma unroll
  for (int q = 0; q < NR; ++q) frag(0, 0, q, fa[0], fb[0]);

  int s = 0;
  for (int ti = 0; ti < my_tiles; ++ti) {
    int tm, tn;
    gemm_tile_of((int)blockIdx.x + ti * (int)gridDim.x, n_tiles, tiles_m, tiles_n, tm, tn, g.group);
    const int m0 = tm * BM, n0 = tn * BN;

    f32x4 acc[FN][FM];
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int i = 0; i < FM; ++i) acc[j][i] = f32x4{};

    // One K step; in the tile's last step (LAST) the fragments of the next
    // tile's first group are read after the epilogue instead (fewer live
    // registers there).
    // With three stages the barrier leaves the DMA of step s + 2 in flight,
    // except in a tile's first step: the previous tile's epilogue stores were
    // issued after that DMA, and the barrier then waits for everything.
    auto step = [&](auto lastc, bool first) {
      constexpr bool LAST = decltype(lastc)::value;
      static_for<2>([&](auto gc) {
        constexpr int gi = decltype(gc)::value;
        if constexpr (gi == 1) {
          if (NS == 2 || first)
            ring_barrier<0>();
          else
            ring_barrier<LPW * (NS - 2)>();
        }
        __builtin_amdgcn_sched_barrier(0);
        static_for<NQ>([&](auto qc) {
          constexpr int q = decltype(qc)::value;
          if constexpr (AMAJ) {
            // A-major order: A fragment i feeds MFMAs i*FN .. i*FN + FN-1 and
            // is then reloaded in place with the next group's fragment i;
            // the W fragments are double-buffered and read at q = i*FN + 1
            // for i < FN.
            constexpr int i = q / FN, j = q % FN;
            acc[j][i] = Mfma16<T>::mma(fb[gi][j], fa[0][i], acc[j][i]);
            if constexpr (gi == 0 || !LAST) {
              constexpr int ng = 1 - gi;  // the next group's index in its step
              const int ns = gi == 0 ? s : s + 1;
              if constexpr (j == 1 % FN && i < FN) frag(ns, ng, i == 0 ? 0 : FM + i, fa[0], fb[ng]);
              if constexpr (j == FN - 1) frag(ns, ng, 1 + i, fa[0], fb[ng]);
            }
          } else {
            constexpr int j = q / FM, i = q % FM;
            acc[j][i] = Mfma16<T>::mma(fb[gi][j], fa[gi][i], acc[j][i]);
#pragma unroll
            for (int r = 0; r < NR; ++r) {
              if (q == r * NQ / NR) {
                if constexpr (gi == 0) frag(s, 1, r, fa[1], fb[1]);
                else if constexpr (!LAST) frag(s + 1, 0, r, fa[0], fb[0]);
              }
            }
          }
          if constexpr (gi == 1) {
#pragma unroll
            for (int d = 0; d < LPW; ++d)
              if (q == d * (NQ / 2) / LPW) dma(s + NS, d);
          }
          __builtin_amdgcn_sched_barrier(0);
        });
      });
      ++s;
    };
    for (int kt = 0; kt + 1 < KT; ++kt) step(std::false_type{}, kt == 0);
    step(std::true_type{}, KT == 1);

    {
      // The lane's position, re-derived per tile behind an opaque copy: the
      // compiler would otherwise hoist every lane-dependent epilogue address
      // out of the tile loop and keep (or spill) them across the K loop.
      int eln = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
      asm volatile("" : "+v"(eln));
      const int lane = eln, fr = eln & 15, kh = eln >> 4;
      (void)lane; (void)fr; (void)kh;
      // ---- epilogue: acc[j][i][e] is output row m0 + wm*TM + 16i + fr,
      // column n0 + wn*TN + 16j + 4kh + e.  Every read (bias, residual rows,
      // row flags) is consumed before the next tile's K loop: a read left
      // pending there would make the compiler wait for it (vmcnt) inside that
      // loop, which also drains the DMA ring.  Accumulator indices are
      // compile-time constants (a runtime index would put acc in scratch).
      int valid[FM];
#pragma unroll
      for (int i = 0; i < FM; ++i)
        valid[i] = QKV || gemm_row_valid(g, min(m0 + wm * TM + 16 * i + fr, g.m - 1));
#pragma unroll
      for (int i = 0; i < FM; ++i) settle(valid[i]);
      typename Raw4<TB>::type braw[FN];
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        braw[j] = {};
        if (epi & TX_EPI_BIAS) braw[j] = ld_raw4(bias + min(n0 + wn * TN + 16 * j + 4 * kh, g.n - 4));
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) settle(braw[j]);
      // Output block (j, i) straight from the MFMA layout: four columns per lane.
      auto direct = [&](auto jc, auto ic, const float* rv) {
        constexpr int j = decltype(jc)::value, i = decltype(ic)::value;
        const int n = n0 + wn * TN + 16 * j + 4 * kh, m = m0 + wm * TM + 16 * i + fr;
        if (n < g.n && m < g.m) {
          float bv[4], a4[4];
          unpack4<TB>(braw[j], bv);
#pragma unroll
          for (int e = 0; e < 4; ++e) a4[e] = acc[j][i][e];
          gemm_finish4<TC, QKV>(g, m, n, a4, bv, rv, valid[i] != 0);
        }
      };
      bool staged = false;
      if constexpr (sizeof(TC) == 2) staged = g.stage16 != 0;
      if (!staged) {
        static_for<FN>([&](auto jc) {
          constexpr int j = decltype(jc)::value;
          typename Raw4<TR>::type rraw[FM];
          const int nc = min(n0 + wn * TN + 16 * j + 4 * kh, g.n - 4);
#pragma unroll
          for (int i = 0; i < FM; ++i) {
            rraw[i] = {};
            if (!QKV && (epi & TX_EPI_RESIDUAL))
              rraw[i] = ld_raw4(res + (int64_t)min(m0 + wm * TM + 16 * i + fr, g.m - 1) * g.ldr + nc);
          }
#pragma unroll
          for (int i = 0; i < FM; ++i) settle(rraw[i]);
          static_for<FM>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            float rv[4];
            unpack4<TR>(rraw[i], rv);
            direct(jc, ic, rv);
          });
        });
      } else if constexpr (sizeof(TC) == 2) {
        // Staged through this wave's LDS region, 16 rows at a time: the rounded
        // (bias, GELU) values go in row-major order, then each lane takes eight
        // consecutive columns of one row -- residual read, residual and mask
        // applied, C written -- as 16-byte accesses (full 128-byte lines where
        // a row segment spans one), instead of 8-byte accesses spread over 16
        // rows.  V columns of the packed-QKV projection keep the direct path
        // (they are written transposed).
        // The residual and the plain epilogues are separate instantiations:
        // with the residual loads under a runtime condition the compiler
        // cannot count the loads in flight and waits for every outstanding
        // memory operation (the next tile's DMA and the previous chunks'
        // stores) before each 16-byte store.
        auto staged_epi = [&](auto resc_c) {
          constexpr int G = TN / 8, SLOTS = 16 * G, PASSES = (SLOTS + 63) / 64;
          TC* stg = reinterpret_cast<TC*>(lds + NS * STAGE) + wave * 16 * ES;
          const TC* __restrict__ resc = reinterpret_cast<const TC*>(g.res);
          TC* __restrict__ C = reinterpret_cast<TC*>(g.c);
          constexpr bool use_res = decltype(resc_c)::value;
          // Residual rows are requested RD - 1 chunks ahead of their use: every
          // chunk at once where that takes at most 32 registers (128-wide
          // tiles), otherwise one chunk ahead.
          constexpr int RD = FM * PASSES * 4 <= 32 ? FM : 2;
          u32x4 rres[use_res ? RD : 1][PASSES];
          auto load_res = [&](int i, u32x4* rr) {
#pragma unroll
            for (int p = 0; p < PASSES; ++p) {
              const int slot = min(64 * p + lane, SLOTS - 1), r = slot / G, c = slot % G;
              const int m = min(m0 + wm * TM + 16 * i + r, g.m - 1), n = min(n0 + wn * TN + 8 * c, g.n - 8);
              rr[p] = u32x4{0u, 0u, 0u, 0u};
              if constexpr (use_res) rr[p] = ld128(resc + (int64_t)m * g.ldr + n);
            }
          };
          if constexpr (use_res) static_for<RD - 1>([&](auto ic) { load_res(decltype(ic)::value, rres[decltype(ic)::value]); });
          static_for<FM>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            __builtin_amdgcn_sched_barrier(0);  // one chunk at a time: bounded live registers
            if constexpr (use_res && i + RD - 1 < FM) load_res(i + RD - 1, rres[(i + RD - 1) % RD]);
            static_for<FN>([&](auto jc) {
              constexpr int j = decltype(jc)::value;
              if (QKV && n0 + wn * TN + 16 * j >= g.qk_cols) return;
              float bv[4], v[4];
              unpack4<TB>(braw[j], bv);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                float t = round_to<TC>(acc[j][i][e] + bv[e]);
                if (epi & TX_EPI_GELU_ERF) t = round_to<TC>(gelu_erf(t));
                v[e] = t;
              }
              st64(stg + fr * ES + 16 * j + 4 * kh, u32x2{pack2<TC>(v[0], v[1]), pack2<TC>(v[2], v[3])});
            });
            // The staging region is private to this wave, and one wave's LDS
            // accesses are performed in issue order: the reads below see the
            // writes above, and the next chunk's writes land after these reads,
            // with no wait.  The empty asm keeps the compiler from reordering
            // the accesses (the 8- and 16-byte views have different types).
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int p = 0; p < PASSES; ++p) {
              const int slot = 64 * p + lane, r = slot / G, c = slot % G;
              const int m = m0 + wm * TM + 16 * i + r, n = n0 + wn * TN + 8 * c;
              const int ok = __shfl(valid[i], r & 15, 64);
              if (slot < SLOTS && m < g.m && n < g.n && !(QKV && n >= g.qk_cols)) {
                u32x4 out = ld128(stg + r * ES + 8 * c);
                if (!QKV && ((epi & (TX_EPI_RESIDUAL | TX_EPI_MASK_OUT)) != 0)) {
                  const u32x4 rw = rres[use_res ? i % RD : 0][p];
                  const bool drop = (epi & TX_EPI_MASK_DELTA) && !ok;
                  const bool zero = (epi & TX_EPI_MASK_OUT) && !ok;
                  float w8[8];
#pragma unroll
                  for (int e = 0; e < 8; ++e) {
                    float t = unpack8<TC>(out, e);
                    if (use_res) t = round_to<TC>(unpack8<TC>(rw, e) + (drop ? 0.f : t));
                    w8[e] = zero ? 0.f : t;
                  }
#pragma unroll
                  for (int e = 0; e < 4; ++e) out[e] = pack2<TC>(w8[2 * e], w8[2 * e + 1]);
                }
                st128(C + (int64_t)m * g.ldc + n, out);
              }
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            if constexpr (QKV) {
              if (g.stage16 & 2) {
                // V columns: the 16 rows of each column go to the staging region
                // transposed (column c at stg + 16 c), then each lane writes eight
                // consecutive sequence positions of one (head, d) row of vt.
                static_for<FN>([&](auto jc) {
                  constexpr int j = decltype(jc)::value;
                  if (n0 + wn * TN + 16 * j < g.qk_cols) return;
                  float bv[4];
                  unpack4<TB>(braw[j], bv);
#pragma unroll
                  for (int e = 0; e < 4; ++e)
                    stg[(16 * j + 4 * kh + e) * 16 + fr] = from_f32<TC>(acc[j][i][e] + bv[e]);
                });
                asm volatile("" ::: "memory");
                __builtin_amdgcn_wave_barrier();
                const int mb = m0 + wm * TM + 16 * i;
                const int bq = mb / g.seq, s0 = mb - bq * g.seq;
#pragma unroll
                for (int p = 0; p < (2 * TN + 63) / 64; ++p) {
                  const int slot = 64 * p + lane, c = slot >> 1, h = slot & 1;
                  const int n = n0 + wn * TN + c;
                  if (slot < 2 * TN && n < g.n && n >= g.qk_cols && mb < g.m) {
                    const int nv = n - g.qk_cols, hh = nv / g.head_dim, d = nv - hh * g.head_dim;
                    TC* dst = reinterpret_cast<TC*>(g.vt) +
                              ((int64_t)(bq * g.heads + hh) * g.head_dim + d) * g.ldvt + s0 + 8 * h;
                    st128(dst, ld128(stg + c * 16 + 8 * h));
                  }
                }
                asm volatile("" ::: "memory");
                __builtin_amdgcn_wave_barrier();
              } else {
                static_for<FN>([&](auto jc) {
                  if (n0 + wn * TN + 16 * decltype(jc)::value >= g.qk_cols) {
                    const float rv[4] = {0.f, 0.f, 0.f, 0.f};
                    direct(jc, ic, rv);
                  }
                });
              }
            }
          });
        };
        if (!QKV && (epi & TX_EPI_RESIDUAL))
          staged_epi(std::true_type{});
        else
          staged_epi(std::false_type{});
      }
    }
    // The next tile's first fragments (its step is stage s % NS).
#pragma unroll
    for (int q = 0; q < NR; ++q) frag(s, 0, q, fa[0], fb[0]);
  }
  ring_drain();
}

// ============================================================ skinny M
// gemm_skinny_kernel: small M where K is not a multiple of 32 (otherwise
// gemm_lsu_kernel runs).  One wave owns a 32 x 32 output block and streams
// its operand fragments straight from global memory into registers (a ring
// PF k-steps deep, no LDS).  KSPLIT = 1: the wave runs the whole K in order
// (bit-identical to the other kernels).  KSPLIT > 1 (variant 9, for
// comparison only): the workgroup's KSPLIT waves each run one K/KSPLIT slice
// and the partial sums are added in slice order through LDS.
template <typename T, typename TC, typename TB, typename TR, int KSPLIT, bool QKV>
__global__ __launch_bounds__(64 * KSPLIT) void gemm_skinny_kernel(GemmArgs g) {
  typedef typename Mfma<T>::vec vec;
  constexpr int PF = 8;
  __shared__ float red[KSPLIT > 1 ? (KSPLIT - 1) * 64 * 16 : 1];
  const int tiles_n = (g.n + 31) / 32;
  const int m0 = (blockIdx.x / tiles_n) * 32, n0 = (blockIdx.x % tiles_n) * 32;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int fr = lane & 31, half = lane >> 5;
  const int kslice = g.k / KSPLIT;
  const int k0 = wave * kslice;
  const int nk = kslice / 16;
  const T* __restrict__ arow = (const T*)g.a + (int64_t)min(m0 + fr, g.m - 1) * g.lda + k0 + 8 * half;
  const T* __restrict__ wrow = (const T*)g.w + (int64_t)min(n0 + fr, g.n - 1) * g.ldw + k0 + 8 * half;

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  vec ab[PF], bb[PF];
#pragma unroll
  for (int i = 0; i < PF; ++i) {
    if (i < nk) {
      ab[i] = __builtin_bit_cast(vec, ld128(arow + 16 * i));
      bb[i] = __builtin_bit_cast(vec, ld128(wrow + 16 * i));
    }
  }
  // Epilogue reads (bias, residual, row flag) go out behind the first
  // operand fragments and land during the K loop.  Addresses are clamped;
  // values past the edge are never stored.
  const TB* __restrict__ bias = (const TB*)g.bias;
  const TR* __restrict__ res = (const TR*)g.res;
  const int m = m0 + fr;
  typename Raw4<TB>::type braw[4];
  typename Raw4<TR>::type rraw[4];
  bool valid = true;
  if (wave == 0) {
    const int mc = min(m, g.m - 1);
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int nc = min(n0 + 8 * q4 + 4 * half, g.n - 4);
      braw[q4] = {};
      rraw[q4] = {};
      if (g.epi & TX_EPI_BIAS) braw[q4] = ld_raw4(bias + nc);
      if (!QKV && (g.epi & TX_EPI_RESIDUAL)) rraw[q4] = ld_raw4(res + (int64_t)mc * g.ldr + nc);
    }
    valid = QKV || gemm_row_valid(g, mc);
  }
  for (int j0 = 0; j0 < nk; j0 += PF) {
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      const int j = j0 + i;
      if (j < nk) {
        acc = Mfma<T>::mma32(bb[i], ab[i], acc);
        if (j + PF < nk) {
          ab[i] = __builtin_bit_cast(vec, ld128(arow + 16 * (j + PF)));
          bb[i] = __builtin_bit_cast(vec, ld128(wrow + 16 * (j + PF)));
        }
      }
    }
  }
  if constexpr (KSPLIT > 1) {
    if (wave > 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) red[((wave - 1) * 16 + r) * 64 + lane] = acc[r];
    }
    __syncthreads();
    if (wave > 0) return;
    // Partials in slice order; two slices per iteration keep the LDS reads
    // in flight without holding every partial in registers at once.
#pragma unroll 2
    for (int w = 1; w < KSPLIT; ++w)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] += red[((w - 1) * 16 + r) * 64 + lane];
  }
  // acc[4*q4 + e]: row m0 + fr, column n0 + 8*q4 + 4*half + e.
  if (m >= g.m) return;
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4) {
    const int n = n0 + 8 * q4 + 4 * half;
    if (n >= g.n) continue;
    float bv[4], rv[4];
    unpack4<TB>(braw[q4], bv);
    unpack4<TR>(rraw[q4], rv);
    float a4[4] = {acc[4 * q4 + 0], acc[4 * q4 + 1], acc[4 * q4 + 2], acc[4 * q4 + 3]};
    gemm_finish4<TC, QKV>(g, m, n, a4, bv, rv, valid);
  }
}

// ------------------------------------------------------------------ launch
// ============================================================ 16 x 16 blocks
// gemm_lsu_kernel: small M (c2's M = 64, the fp32-model c1's 256) on
// v_mfma_f32_16x16x32: one 16 x 16 output block per workgroup of NW waves.
// 16-row blocks give four times as many waves as 32 x 32 blocks, and each
// MFMA covers 32 values of K, so a wave's K loop has half as many dependent
// steps; operand fragments stream from global memory into a register ring
// (no LDS).
//  NW = 1: the wave runs the whole K in order (bit-identical to the in-order
//   kernels above).
//  NW = 4 (K >= 2048): the library's kernel at these shapes (MT16x16x128 with
//   four local split-K waves) fixes the accumulation order, and this
//   reproduces it: wave w accumulates, for each 128-deep block i of K in
//   ascending order, the 32-deep chunk [128 i + 32 w, 128 i + 32 w + 32); the
//   four partials are added in wave order, ((p0 + p1) + p2) + p3.

template <typename T, typename TC, typename TB, typename TR, bool QKV, int NW = 4>
__global__ __launch_bounds__(64 * NW) void gemm_lsu_kernel(GemmArgs g) {
  typedef typename Mfma16<T>::vec vec;
  // Fragments in flight: all of K at c2's shapes (K / 32 / NW = 16), so the
  // loop waits for one memory latency.
  constexpr int PF = 16;
  __shared__ float red[NW > 1 ? (NW - 1) * 4 * 64 : 1];
  const int tiles_n = (g.n + 15) / 16;
  const int m0 = (blockIdx.x / tiles_n) * 16, n0 = (blockIdx.x % tiles_n) * 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // 16x16x32 operands: lane l holds row (l & 15), k = 8 (l >> 4) .. +7 of the
  // chunk.  D^T = W A^T: lane l gets output row m0 + (l & 15) and the four
  // consecutive columns n0 + 4 (l >> 4) + e.
  const int fr = lane & 15, kg = lane >> 4;
  constexpr int KST = 32 * NW;  // k stride between a wave's chunks
  const int nk = g.k / KST;
  const T* __restrict__ arow = (const T*)g.a + (int64_t)min(m0 + fr, g.m - 1) * g.lda + 32 * wave + 8 * kg;
  const T* __restrict__ wrow = (const T*)g.w + (int64_t)min(n0 + fr, g.n - 1) * g.ldw + 32 * wave + 8 * kg;
  // The epilogue's reads (bias, residual, row flag; clamped into the operands)
  // go out first: they do not depend on the products, so their latency
  // overlaps the K loop instead of following it.  The residual may alias C:
  // this block is read here before any of it is written.
  const int m = m0 + fr, n = n0 + 4 * kg;
  const int mc = min(m, g.m - 1), nc = min(n, g.n - 4);
  typename Raw4<TB>::type braw = {};
  typename Raw4<TR>::type rraw = {};
  bool valid = true;
  if (wave == 0) {
    if (g.epi & TX_EPI_BIAS) braw = ld_raw4((const TB*)g.bias + nc);
    if (!QKV && (g.epi & TX_EPI_RESIDUAL)) rraw = ld_raw4((const TR*)g.res + (int64_t)mc * g.ldr + nc);
    valid = QKV || gemm_row_valid(g, mc);
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  vec ab[PF], bb[PF];
#pragma unroll
  for (int i = 0; i < PF; ++i)
    if (i < nk) {
      ab[i] = __builtin_bit_cast(vec, ld128(arow + KST * i));
      bb[i] = __builtin_bit_cast(vec, ld128(wrow + KST * i));
    }
  for (int j0 = 0; j0 < nk; j0 += PF) {
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      const int j = j0 + i;
      if (j < nk) {
        acc = Mfma16<T>::mma(bb[i], ab[i], acc);
        if (j + PF < nk) {
          ab[i] = __builtin_bit_cast(vec, ld128(arow + KST * (j + PF)));
          bb[i] = __builtin_bit_cast(vec, ld128(wrow + KST * (j + PF)));
        }
      }
    }
  }
  if constexpr (NW > 1) {
    if (wave > 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) red[((wave - 1) * 4 + r) * 64 + lane] = acc[r];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 1; w < NW; ++w)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] += red[((w - 1) * 4 + r) * 64 + lane];
  }
  if (m >= g.m || n >= g.n) return;
  float bv[4], rv[4];
  unpack4<TB>(braw, bv);
  unpack4<TR>(rraw, rv);
  float a4[4] = {acc[0], acc[1], acc[2], acc[3]};
  gemm_finish4<TC, QKV>(g, m, n, a4, bv, rv, valid);
}

struct TileCfg {
  int bm, bn;
};

template <typename T, typename TC, typename TB, typename TR, bool QKV>
static int launch_gemm_small(const GemmArgs& g, hipStream_t st) {
  // 128x128 when that still gives every CU a tile, else 64x64.  (The
  // register-staged kernel's 256-row tiles need more than 256 VGPRs and
  // spill; shapes large enough for them take gemm_big_kernel whenever K is a
  // multiple of 64.)
  static const TileCfg cfgs[] = {{128, 128}, {64, 64}};
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  int pick = 1;
  for (int c = 0; c < 2; ++c) {
    const long tiles = (long)((g.m + cfgs[c].bm - 1) / cfgs[c].bm) * ((g.n + cfgs[c].bn - 1) / cfgs[c].bn);
    if (tiles >= cus) {
      pick = c;
      break;
    }
  }
  const long tiles = (long)((g.m + cfgs[pick].bm - 1) / cfgs[pick].bm) *
                     ((g.n + cfgs[pick].bn - 1) / cfgs[pick].bn);
  if (tiles > 0x7fffffffL) return TX_EUNSUPPORTED;
  dim3 grid((unsigned)tiles);
  if (pick == 0)
    gemm_kernel<T, TC, TB, TR, 128, 128, 2, 2, QKV><<<grid, dim3(256), 0, st>>>(g);
  else
    gemm_kernel<T, TC, TB, TR, 64, 64, 2, 2, QKV><<<grid, dim3(256), 0, st>>>(g);
  return hipGetLastError() == hipSuccess ? TX_OK : TX_EHIP;
}

template <typename T, typename TC, typename TB, typename TR, int BM, int BN, int BK, int WM, int WN,
          int STAGES, int OPT, bool QKV>
static int launch_big(const GemmArgs& g, hipStream_t st) {
  const long tiles = (long)((g.m + BM - 1) / BM) * ((g.n + BN - 1) / BN);
  if (tiles > 0x7fffffffL) return TX_EUNSUPPORTED;
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const long slots = (long)cus * big_per_cu<T, BM, BN, BK, STAGES>();
  const long grid = tiles < slots ? tiles : slots;
  gemm_big_kernel<T, TC, TB, TR, BM, BN, BK, WM, WN, STAGES, OPT, QKV>
      <<<dim3((unsigned)grid), dim3(WM * WN * 64), 0, st>>>(g);
  return hipGetLastError() == hipSuccess ? TX_OK : TX_EHIP;
}

template <typename T> constexpr int dt_code() {
  return std::is_same<T, float>::value ? TX_F32 : std::is_same<T, f16>::value ? TX_F16 : TX_BF16;
}

static inline bool al(const void* p, int bytes) { return ((uintptr_t)p % bytes) == 0; }

template <typename T, typename TC, typename TB, typename TR, int BN, bool QKV, int NS = 2>
static int launch_hp(const GemmArgs& g0, hipStream_t st) {
  GemmArgs g = g0;
  // Staged (16-byte) epilogue: 16-bit C and residual, rows of whole 8-column
  // groups, 16-byte aligned (TX_GEMM_STAGE=0 turns it off; tuning only).
  static const bool stage_env = [] {
    const char* e = getenv("TX_GEMM_STAGE");
    return !(e && e[0] == '0');
  }();
  g.stage16 = (stage_env && sizeof(TC) == 2 && !(g.epi & TX_EPI_SPLIT_OUT) && g.n % 8 == 0 &&
               g.ldc % 8 == 0 && al(g.c, 16) && (!QKV || g.qk_cols % 8 == 0) &&
               (!(g.epi & TX_EPI_RESIDUAL) || (g.ldr % 8 == 0 && al(g.res, 16))))
                  ? 1
                  : 0;
  // Packed-QKV V columns staged too when every 16-row chunk lies in one
  // sequence and every 16-column block in one head, with 16-byte vt rows.
  if (QKV && g.stage16 && g.seq % 16 == 0 && g.m % 16 == 0 && g.head_dim % 16 == 0 && g.ldvt % 8 == 0 &&
      g.qk_cols % 16 == 0 && al(g.vt, 16))
    g.stage16 |= 2;
  const long tiles = (long)((g.m + 255) / 256) * ((g.n + BN - 1) / BN);
  if (tiles > 0x7fffffffL) return TX_EUNSUPPORTED;
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const long grid = tiles < cus ? tiles : cus;
  gemm_hp_kernel<T, TC, TB, TR, BN, QKV, NS><<<dim3((unsigned)grid), dim3(512), 0, st>>>(g);
  return hipGetLastError() == hipSuccess ? TX_OK : TX_EHIP;
}

template <typename T, typename TC, typename TB, typename TR, bool QKV>
static int launch_gemm_typed(const GemmArgs& g0, hipStream_t st) {
  GemmArgs g = g0;
  // Tile rows per band of the persistent kernels' tile order (TX_GEMM_GROUP
  // overrides; tuning only).
  static const int group_env = [] {
    const char* e = getenv("TX_GEMM_GROUP");
    return e ? atoi(e) : 0;
  }();
  g.group = group_env > 0 ? group_env : 8;
  // Big-tile path: K a multiple of 64, at least one 256-row tile, vector
  // alignment of C / residual for the 4-column epilogue.
  const bool vec_ok = (g.n % 4 == 0) && (g.ldc % 4 == 0) && al(g.c, 4 * sizeof(TC)) &&
                      (!(g.epi & TX_EPI_BIAS) || al(g.bias, 4 * sizeof(TB))) &&
                      (!(g.epi & TX_EPI_RESIDUAL) || ((g.ldr % 4 == 0) && al(g.res, 4 * sizeof(TR))));
  // Tile shape: gemm_hp_kernel (256 x BN, eight waves, hand-ordered
  // pipeline) with BN from gemm_hp_width.  A/B in one process against
  // gemm_big_kernel's 128x128 tiles (2x2 waves of 64x64, two workgroups per
  // CU) and 256x256 tiles (2x4 waves of 128x64): 8-23% faster at every c3/c4
  // shape.  Measured and not chosen (hp kernel): four waves of 128x128 /
  // 128 x BN/2 (one wave per SIMD: 10-60% slower, waits exposed), 32x32x16
  // MFMAs (5-10% slower), BK = 32 with four stages (half-line L2 requests,
  // slower), fragment reads packed at the start of a group (3-5% slower).
  // tx_select_kernel / TX_GEMM_VARIANT override the choice (tests and timing):
  // 0 gemm_kernel; 8, 9 gemm_skinny_kernel; 10, 11 gemm_lsu_kernel; 19, 20
  // gemm_big_kernel; 128 to 256, 1283 gemm_hp_kernel; 1000 + i gemm_ring_kernel's
  // configuration i.  Where one does not take the shape: gemm_kernel.
  int variant = selected_kernel(TX_SELECT_GEMM);
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const long t256 = (long)((g.m + 255) / 256) * ((g.n + 255) / 256);
  // Skinny M: fewer 256-row tiles than CUs and at most 256 rows.  K below
  // 2048 runs in order on one wave per 16x16 block (gemm_lsu_kernel, NW = 1);
  // K >= 2048 (a multiple of 128) runs the library's local split-K order
  // over four waves (NW = 4), bit-identical to F.linear at e.g. M = 64,
  // K = 2048; K % 32 == 16 takes the in-order 32x32 skinny kernel.
  const bool skinny_ok = vec_ok && g.m <= 256 && t256 < cus && g.k % 16 == 0;
  // The library splits K over four waves at small M and K >= 2048 (NW = 4
  // reproduces that order); everywhere else it accumulates in order.
  const bool lsu4 = g.k >= 2048 && g.k % 128 == 0;
  // gemm_ring_kernel: K a multiple of 64 (64-bit row strides excluded).
  const bool ring_ok = vec_ok && g.k % 64 == 0 && hp_offsets_fit(g.lda, g.ldw, g.k, sizeof(T));
  auto ring = [&](int cfg, bool ks4) {
    return launch_gemm_ring(g, dt_code<T>(), dt_code<TC>(), dt_code<TR>(), QKV, cfg, ks4, st);
  };
  double ring_us = 0.0;
  const bool ring_ks4 = skinny_ok && lsu4;
  const int ring_cfg = gemm_ring_pick(g.m, g.n, g.k, g.epi & TX_EPI_GELU_ERF, cus, ring_ks4, &ring_us);
  if (variant >= 1000 && variant < 1006 && ring_ok) return ring(variant - 1000, ring_ks4 && variant < 1002);
  // Small M: 16 x 16 blocks while they are few (c2's shapes: 64x1536x512 4.9
  // against 5.3 us), ring tiles (same bits) where the blocks' operand reads
  // grow past them (190x2048x2048 25.3 against 10.6 us, 102x3072x1024 14.2
  // against 8.2).  Modelled times in us, fitted to 60 random shapes with
  // M 17 .. 256 (within 10%): a base, the chain over K, and the operand reads
  // of all blocks.
  if (skinny_ok && ring_ok && variant < 0) {
    const double reads = (double)((g.m + 15) / 16) * ((g.n + 15) / 16) * g.k;
    const double lsu_us = lsu4 ? 4.06 + 2.67e-4 * g.k + 6.4e-6 * reads : 2.98 + 8.07e-4 * g.k + 6.8e-6 * reads;
    if (ring_us < lsu_us) return ring(ring_cfg, ring_ks4);
  }
  if (skinny_ok && g.k % 32 == 0 && ((variant < 0 && !lsu4) || variant == 11)) {
    const long blocks = (long)((g.m + 15) / 16) * ((g.n + 15) / 16);
    gemm_lsu_kernel<T, TC, TB, TR, QKV, 1><<<dim3((unsigned)blocks), dim3(64), 0, st>>>(g);
    return hipGetLastError() == hipSuccess ? TX_OK : TX_EHIP;
  }
  if (skinny_ok && g.k % 128 == 0 && ((variant < 0 && lsu4) || variant == 10)) {
    const long blocks = (long)((g.m + 15) / 16) * ((g.n + 15) / 16);
    gemm_lsu_kernel<T, TC, TB, TR, QKV><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(g);
    return hipGetLastError() == hipSuccess ? TX_OK : TX_EHIP;
  }
  if (skinny_ok && (variant < 0 || variant == 8 || variant == 9)) {
    const long blocks = (long)((g.m + 31) / 32) * ((g.n + 31) / 32);
    const bool split = (variant == 9);
    if (split && g.k % 128 == 0)
      gemm_skinny_kernel<T, TC, TB, TR, 8, QKV><<<dim3((unsigned)blocks), dim3(512), 0, st>>>(g);
    else
      gemm_skinny_kernel<T, TC, TB, TR, 1, QKV><<<dim3((unsigned)blocks), dim3(64), 0, st>>>(g);
    return hipGetLastError() == hipSuccess ? TX_OK : TX_EHIP;
  }
  const bool big_ok = g.k % 64 == 0 && g.m >= 256 && vec_ok;
  if (!big_ok || variant == 0) return launch_gemm_small<T, TC, TB, TR, QKV>(g, st);
  if (variant < 0) {
    GemmShape s{};
    s.m = g.m;
    s.n = g.n;
    s.k = g.k;
    s.gelu = g.epi & TX_EPI_GELU_ERF;
    s.residual = g.epi & TX_EPI_RESIDUAL;
    s.split = !QKV && (g.epi & TX_EPI_SPLIT_OUT);
    s.f32 = sizeof(TC) == 4 && !s.split;
    s.qkv = QKV;
    s.seq = g.seq;
    variant = gemm_route(s, cus, ring_ok);
    if (variant >= 1000) return ring(variant - 1000, false);
  }
  // gemm_hp_kernel's per-lane DMA offsets are 32-bit (hp_offsets_fit); wider
  // row strides take the 128x128 kernel, which addresses in 64 bits.
  // 128-wide tiles run with three K stages (their three stages fit in LDS):
  // inside the forward, where operands come from HBM or the MALL rather than
  // a warm L2, the extra step of DMA lookahead took c3 from 1.952 to 1.827
  // ms (A/B on one box; the same launches repeated in isolation: within 3%).
  // TX_GEMM_HP3=0 keeps two stages (tuning only).
  static const bool hp3_env = [] {
    const char* e = getenv("TX_GEMM_HP3");
    return !(e && e[0] == '0');
  }();
  if (variant == 128 && hp3_env) variant = 1283;
  if ((variant == 256 || variant == 192 || variant == 128 || variant == 1283) &&
      !hp_offsets_fit(g.lda, g.ldw, g.k, sizeof(T)))
    variant = 20;
  switch (variant) {
    case 19: return launch_big<T, TC, TB, TR, 256, 256, 64, 2, 4, 2, 6, QKV>(g, st);
    case 20: return launch_big<T, TC, TB, TR, 128, 128, 64, 2, 2, 2, 6, QKV>(g, st);
    case 256: return launch_hp<T, TC, TB, TR, 256, QKV>(g, st);
    case 192: return launch_hp<T, TC, TB, TR, 192, QKV>(g, st);
    case 128: return launch_hp<T, TC, TB, TR, 128, QKV>(g, st);
    case 1283: return launch_hp<T, TC, TB, TR, 128, QKV, 3>(g, st);
    default: return launch_gemm_small<T, TC, TB, TR, QKV>(g, st);
  }
}

int launch_gemm(const GemmArgs& g, int ab_dt, int c_dt, int bias_dt, int res_dt, bool qkv,
                hipStream_t st) {
  if (bias_dt != ab_dt) return TX_EUNSUPPORTED;
  if (ab_dt == TX_BF16) {
    if (c_dt == TX_BF16 && res_dt == TX_BF16)
      return qkv ? launch_gemm_typed<bf16, bf16, bf16, bf16, true>(g, st)
                 : launch_gemm_typed<bf16, bf16, bf16, bf16, false>(g, st);
    if (qkv) return TX_EUNSUPPORTED;
    if (c_dt == TX_F32 && res_dt == TX_F32) return launch_gemm_typed<bf16, float, bf16, float, false>(g, st);
    if (c_dt == TX_F32 && res_dt == TX_BF16) return launch_gemm_typed<bf16, float, bf16, bf16, false>(g, st);
  }
  if (ab_dt == TX_F16) {
    if (c_dt == TX_F16 && res_dt == TX_F16)
      return qkv ? launch_gemm_typed<f16, f16, f16, f16, true>(g, st)
                 : launch_gemm_typed<f16, f16, f16, f16, false>(g, st);
    if (qkv) return TX_EUNSUPPORTED;
    if (c_dt == TX_F32 && res_dt == TX_F32) return launch_gemm_typed<f16, float, f16, float, false>(g, st);
    if (c_dt == TX_F32 && res_dt == TX_F16) return launch_gemm_typed<f16, float, f16, f16, false>(g, st);
  }
  return TX_EUNSUPPORTED;
}

}  // namespace tx
