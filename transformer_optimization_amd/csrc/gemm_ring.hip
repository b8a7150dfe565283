// gemm_ring_kernel: tiles of 64 to 128 rows.  First of all for outputs with too
// few 256-row tiles to fill the CUs (the reference CLI's default shape, B8 S128
// D512 F2048, gives gemm_hp_kernel 16 to 64 tiles on 256 CUs), and for any other
// whose modelled time is less (gemm_route.hpp), up to 100000 rows.
//
// One workgroup of eight waves (2 x 4) per BM x BN tile (64 to 192 columns), not
// persistent: with two workgroups per CU one's epilogue and first loads run
// beside the other's K loop.  K advances in steps of 64 through NS LDS stages
// fed by global_load_lds_dwordx4.
//
// What bounds it: at few tiles waits (waves wait half of their life at 1024 rows,
// vector and matrix pipes both far from busy): the first loads, the LDS port in
// the K step (a 64 x 64 step moves 48 KB of fragments and 16 KB of DMA; eight
// stages instead of four took 9.6 against 9.3 us at 1024x512x2048, so it is not
// the bytes in flight), and CUs without a tile.  On full grids the matrix cores
// are 0.3 to 0.42 busy and, with GELU, the vector ALUs 0.38 to 0.52.
//
// Inside a step, as in gemm_hp_kernel: the MFMAs (v_mfma_f32_16x16x32) of
// k32 group 0 with the fragment reads of group 1 between them; the wait for
// step s + 1 and one barrier; the MFMAs of group 1 with the fragment reads of
// step s + 1's group 0 and the DMA issues of step s + NS between them.  No
// step past the last is issued (at K = 512 they would be half of the
// traffic), so the last NS - 1 steps wait with their own counts.
//
// Per output element the products are accumulated with k ascending in one
// chain, as in the other in-order kernels: identical bits.
#include <cstdlib>

#include "common.hpp"
#include "gemm_common.hpp"
#include "tx_internal.hpp"

namespace tx {

// Wait until at most LPW * rem of this wave's DMA issues are in flight (rem
// wave-uniform, 0 .. MAX), then barrier.
template <int LPW, int MAX>
__device__ __forceinline__ void ring_wait(int rem) {
  static_for<MAX + 1>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    if (rem == j) ring_barrier<LPW * j>();
  });
}

//
// KS4 reproduces gemm_lsu_kernel's four-wave order instead (the library's
// local split of K at M <= 256, K >= 2048): the 32-deep chunk w of every
// 128-deep block of K goes to accumulator set w, in order, and the four sums
// are added in order of w.  K is then a multiple of 128.
template <typename T, typename TC, typename TB, typename TR, int BM, int BN, int NS, bool QKV, bool KS4>
__global__ __launch_bounds__(512) void gemm_ring_kernel(GemmArgs g) {
  constexpr int WM = 2, WN = 4;  // eight waves
  constexpr int BK = 64, NW = WM * WN, NT = NW * 64;
  constexpr int RPI = 8;  // LDS rows (128 bytes) filled by one DMA instruction
  constexpr int TM = BM / WM, TN = BN / WN;
  constexpr int FM = TM / 16, FN = TN / 16;
  constexpr int A_LD = BM / RPI / NW, B_LD = BN / RPI / NW, LPW = A_LD + B_LD;
  constexpr int NR = FM + FN, NQ = FM * FN;
  constexpr int STAGE = (BM + BN) * BK;
  static_assert(A_LD * RPI * NW == BM && B_LD * RPI * NW == BN, "load split");
  static_assert(NS >= 2 && LPW * (NS - 1) <= 63, "vmcnt range");
  static_assert(!KS4 || NS % 2 == 0, "steps in pairs");
  constexpr int NA = KS4 ? 4 : 1;  // accumulator sets
  typedef typename Mfma16<T>::vec vec;
  // Epilogue staging in the ring's memory: C rows of BN values, or (V columns
  // of the packed projection) columns of BM, padded by 16 bytes.
  constexpr int ES = BN + 8, EV = BM + 8;
  static_assert(BM * ES <= NS * STAGE && BN * EV <= NS * STAGE, "staging fits the ring");
  __shared__ __attribute__((aligned(16))) T lds[NS * STAGE];

  const int tiles_m = (g.m + BM - 1) / BM, tiles_n = (g.n + BN - 1) / BN;
  int tm, tn;
  gemm_tile_of((int)blockIdx.x, (int)gridDim.x, tiles_m, tiles_n, tm, tn, g.group);
  const int m0 = tm * BM, n0 = tn * BN;
  const int KT = g.k / BK;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t epi = g.epi;

  // ---- loader: uniform tile bases, per-lane byte offsets; rows past the
  // edge are clamped into the operand (they feed discarded outputs).
  const int lr = lane >> 3, lp = lane & 7;
  const uint32_t chk = (uint32_t)(8 * (lp ^ big_swz<8>(lr)) * (int)sizeof(T));
  const char* abase = (const char*)g.a + (int64_t)m0 * g.lda * (int64_t)sizeof(T);
  const char* bbase = (const char*)g.w + (int64_t)n0 * g.ldw * (int64_t)sizeof(T);
  uint32_t aoff[A_LD], boff[B_LD];
#pragma unroll
  for (int i = 0; i < A_LD; ++i)
    aoff[i] = (uint32_t)(min((i * NW + wave) * RPI + lr, g.m - 1 - m0) * (int)g.lda * (int)sizeof(T)) + chk;
#pragma unroll
  for (int i = 0; i < B_LD; ++i)
    boff[i] = (uint32_t)(min((i * NW + wave) * RPI + lr, g.n - 1 - n0) * (int)g.ldw * (int)sizeof(T)) + chk;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)lds;
  auto dma = [&](int s, int q) {
    const int kb = s * BK * (int)sizeof(T);
    const uint32_t st = lds0 + (uint32_t)((s % NS) * STAGE * (int)sizeof(T));
    if (q < A_LD)
      dma16_m0(abase + kb, aoff[q < A_LD ? q : 0], st + (uint32_t)((q * NW + wave) * RPI * BK * (int)sizeof(T)));
    else
      dma16_m0(bbase + kb, boff[q < A_LD ? 0 : q - A_LD],
               st + (uint32_t)((BM * BK + ((q - A_LD) * NW + wave) * RPI * BK) * (int)sizeof(T)));
  };

  // ---- fragment read q (0 .. NR-1) of k32 group grp of step s, in the order
  // the MFMAs consume them: W fragment 0, the FM A fragments, W fragments 1 ..
  const int wm = wave / WN, wn = wave % WN;
  const int fr = lane & 15, kh = lane >> 4;
  const int fs = big_swz<8>(fr);
  const int a_row = (wm * TM + fr) * BK, b_row = BM * BK + (wn * TN + fr) * BK;
  vec fa[2][FM], fb[2][FN];
  auto frag = [&](int s, int grp, int q, vec* a, vec* b) {
    const T* base = lds + (s % NS) * STAGE + 8 * ((4 * grp + kh) ^ fs);
    if (q == 0) b[0] = *reinterpret_cast<const vec*>(base + b_row);
    else if (q <= FM) a[q - 1] = *reinterpret_cast<const vec*>(base + a_row + 16 * (q - 1) * BK);
    else b[q - FM] = *reinterpret_cast<const vec*>(base + b_row + 16 * (q - FM) * BK);
  };

  // ---- the epilogue's reads (bias, residual, row flags; addresses clamped into
  // the operands) go out first: they do not depend on the products, and at K =
  // 512 their latency after the K loop was a tenth of the launch.  The residual
  // may alias C: each value is read here by the lane that writes it.  (Larger
  // tiles have no registers to hold the residual and read it after the loop.)
  const bool staged = sizeof(TC) == 2 && g.stage16;
  constexpr int CPR = BN / 8, CH = BM * CPR / NT;  // staged: 16-byte chunks per row, per thread
  static_assert(CH * NT == BM * CPR, "chunks per thread");
  constexpr bool PRE_S = CH <= 2, PRE_D = FM * FN <= 4;
  typename Raw4<TB>::type braw[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    braw[j] = {};
    if (epi & TX_EPI_BIAS) braw[j] = ld_raw4((const TB*)g.bias + min(n0 + wn * TN + 16 * j + 4 * kh, g.n - 4));
  }
  u32x4 rres[CH];               // staged
  bool rok[CH];
  typename Raw4<TR>::type rraw[FN][FM];  // direct
  auto load_staged = [&]() {
#pragma unroll
    for (int p = 0; p < CH; ++p) {
      rres[p] = u32x4{0u, 0u, 0u, 0u};
      rok[p] = true;
      if (!QKV && (epi & (TX_EPI_RESIDUAL | TX_EPI_MASK_OUT))) {
        const int ch = p * NT + tid, m = min(m0 + ch / CPR, g.m - 1), n = min(n0 + 8 * (ch % CPR), g.n - 8);
        if (epi & TX_EPI_RESIDUAL) rres[p] = ld128((const TC*)g.res + (int64_t)m * g.ldr + n);
        rok[p] = gemm_row_valid(g, m);
      }
    }
  };
  auto load_direct = [&](int j) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      rraw[j][i] = {};
      if (!QKV && (epi & TX_EPI_RESIDUAL))
        rraw[j][i] = ld_raw4((const TR*)g.res + (int64_t)min(m0 + wm * TM + 16 * i + fr, g.m - 1) * g.ldr +
                             min(n0 + wn * TN + 16 * j + 4 * kh, g.n - 4));
    }
  };
  if constexpr (sizeof(TC) == 2 && PRE_S) {
    if (staged) load_staged();
  }
  if constexpr (PRE_D) {
    if (!staged) {
#pragma unroll
      for (int j = 0; j < FN; ++j) load_direct(j);
    }
  }

  // ---- prologue
  const int pre = min(NS, KT);
#pragma unroll
  for (int s = 0; s < NS; ++s)
    if (s < pre) {
#pragma unroll
      for (int q = 0; q < LPW; ++q) dma(s, q);
    }
  f32x4 accs[NA][FN][FM];
#pragma unroll
  for (int w = 0; w < NA; ++w)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int i = 0; i < FM; ++i) accs[w][j][i] = f32x4{};
  ring_wait<LPW, NS - 1>(pre - 1);
#pragma unroll
  for (int q = 0; q < NR; ++q) frag(0, 0, q, fa[0], fb[0]);

  // KIND 0: steps whose s + NS is still to be issued; 1: the steps after
  // them; 2: the last one.  PAR: s & 1 (KS4).
  auto step = [&](auto kindc, auto parc, int s) {
    constexpr int KIND = decltype(kindc)::value, PAR = decltype(parc)::value;
    static_for<2>([&](auto gc) {
      constexpr int gi = decltype(gc)::value;
      if constexpr (gi == 1) {
        if constexpr (KIND == 0) ring_barrier<LPW * (NS - 2)>();
        if constexpr (KIND == 1) ring_wait<LPW, NS - 2>(KT - 2 - s);
      }
      __builtin_amdgcn_sched_barrier(0);
      static_for<NQ>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        constexpr int j = q / FM, i = q % FM;
        constexpr int w = KS4 ? 2 * PAR + gi : 0;
        accs[w][j][i] = Mfma16<T>::mma(fb[gi][j], fa[gi][i], accs[w][j][i]);
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if (q == r * NQ / NR) {
            if constexpr (gi == 0) frag(s, 1, r, fa[1], fb[1]);
            else if constexpr (KIND != 2) frag(s + 1, 0, r, fa[0], fb[0]);
          }
        if constexpr (gi == 1 && KIND == 0) {
#pragma unroll
          for (int d = 0; d < LPW; ++d)
            if (q == d * NQ / LPW) dma(s + NS, d);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };
  typedef std::integral_constant<int, 0> c0;
  typedef std::integral_constant<int, 1> c1;
  typedef std::integral_constant<int, 2> c2;
  int s = 0;
  if constexpr (KS4) {
    for (; s + NS < KT; s += 2) {
      step(c0{}, c0{}, s);
      step(c0{}, c1{}, s + 1);
    }
    for (; s + 2 < KT; s += 2) {
      step(c1{}, c0{}, s);
      step(c1{}, c1{}, s + 1);
    }
    step(c1{}, c0{}, s);
    step(c2{}, c1{}, s + 1);
  } else {
    for (; s + NS < KT; ++s) step(c0{}, c0{}, s);
    for (; s + 1 < KT; ++s) step(c1{}, c0{}, s);
    step(c2{}, c0{}, s);
  }
  f32x4(&acc)[FN][FM] = accs[0];
  if constexpr (KS4) {
#pragma unroll
    for (int w = 1; w < 4; ++w)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int i = 0; i < FM; ++i) acc[j][i] += accs[w][j][i];
  }

  // ---------------------------------------------------------------- epilogue
  // acc[j][i][e]: row m0 + wm*TM + 16i + fr, column n0 + wn*TN + 16j + 4kh + e.
  if (staged) {
    if constexpr (sizeof(TC) == 2) {
      // Staged through LDS so that C, the residual and V^T move as 16-byte
      // runs of whole rows.
      TC* stg = reinterpret_cast<TC*>(lds);
      TC* __restrict__ C = reinterpret_cast<TC*>(g.c);
      // V columns of this tile start at vc (a multiple of 16: whole 16-column
      // blocks are on one side); q / k columns go first, then V.
      const int vc = QKV ? min(max(g.qk_cols - n0, 0), BN) : BN;
      if constexpr (!PRE_S) load_staged();  // before the rounding and GELU
      __syncthreads();  // every wave has read its last fragments
      if (!QKV || vc > 0) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          float bv[4];
          unpack4<TB>(braw[j], bv);
          if (QKV && wn * TN + 16 * j >= vc) continue;
#pragma unroll
          for (int i = 0; i < FM; ++i) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float t = round_to<TC>(acc[j][i][e] + bv[e]);
              if (epi & TX_EPI_GELU_ERF) t = round_to<TC>(gelu_erf(t));
              v[e] = t;
            }
            st64(stg + (wm * TM + 16 * i + fr) * ES + wn * TN + 16 * j + 4 * kh,
                 u32x2{pack2<TC>(v[0], v[1]), pack2<TC>(v[2], v[3])});
          }
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < CH; ++p) {
          const int ch = p * NT + tid, r = ch / CPR, c = ch % CPR;
          const int m = m0 + r, n = n0 + 8 * c;
          if (m < g.m && n < g.n && (!QKV || 8 * c < vc)) {
            u32x4 out = ld128(stg + r * ES + 8 * c);
            if (!QKV && ((epi & (TX_EPI_RESIDUAL | TX_EPI_MASK_OUT)) != 0)) {
              const bool drop = (epi & TX_EPI_MASK_DELTA) && !rok[p];
              const bool zero = (epi & TX_EPI_MASK_OUT) && !rok[p];
              float w8[8];
#pragma unroll
              for (int e = 0; e < 8; ++e) {
                float t = unpack8<TC>(out, e);
                if (epi & TX_EPI_RESIDUAL) t = round_to<TC>(unpack8<TC>(rres[p], e) + (drop ? 0.f : t));
                w8[e] = zero ? 0.f : t;
              }
#pragma unroll
              for (int e = 0; e < 4; ++e) out[e] = pack2<TC>(w8[2 * e], w8[2 * e + 1]);
            }
            st128(C + (int64_t)m * g.ldc + n, out);
          }
        }
      }
      if (QKV && vc < BN) {
        if (vc > 0) __syncthreads();  // the q / k columns have been read
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int col = wn * TN + 16 * j + 4 * kh;
          float bv[4];
          unpack4<TB>(braw[j], bv);
          if (wn * TN + 16 * j < vc) continue;
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              stg[(col + e) * EV + wm * TM + 16 * i + fr] = from_f32<TC>(acc[j][i][e] + bv[e]);
        }
        __syncthreads();
        // V^T rows: per column, the tile's rows are up to two runs of sequence
        // positions (staged only where seq >= BM), each written as 8-position
        // chunks aligned in the row; partial chunks element by element.
        const int b0 = m0 / g.seq, s0 = m0 - b0 * g.seq;
        const int rows = min(BM, g.m - m0);
        const int len0 = min(rows, g.seq - s0);              // run 0: positions s0 .. s0 + len0 - 1 of b0
        const int c0 = s0 >> 3, nch0 = ((s0 + len0 + 7) >> 3) - c0;
        const int nch = nch0 + ((rows - len0 + 7) >> 3);     // run 1: positions 0 .. rows - len0 - 1 of b0 + 1
        constexpr int MAXC = BM / 8 + 2;
        for (int it = tid; it < (BN - vc) * MAXC; it += NT) {
          const int col = vc + it / MAXC, c = it % MAXC;
          const int n = n0 + col;
          if (n >= g.n || c >= nch) continue;
          const int nv = n - g.qk_cols, hh = nv / g.head_dim, d = nv - hh * g.head_dim;
          const int run = c >= nch0 ? 1 : 0;
          const int p0 = 8 * (run ? c - nch0 : c0 + c);       // the chunk's first position
          const int lo = run ? 0 : s0, hi = run ? rows - len0 : s0 + len0;
          const TC* src = stg + col * EV + (run ? len0 + p0 : p0 - s0);
          TC* dst = (TC*)g.vt + ((int64_t)((b0 + run) * g.heads + hh) * g.head_dim + d) * g.ldvt + p0;
          if (p0 >= lo && p0 + 8 <= hi) {
            u32x4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e)
              w[e] = (uint32_t)__builtin_bit_cast(uint16_t, src[2 * e]) |
                     ((uint32_t)__builtin_bit_cast(uint16_t, src[2 * e + 1]) << 16);
            st128(dst, w);
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (p0 + e >= lo && p0 + e < hi) dst[e] = src[e];
          }
        }
      }
      return;
    }
  }
  // fp32 or split outputs, and rows without 16-byte alignment: four columns
  // per lane straight from the MFMA layout.
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int n = n0 + wn * TN + 16 * j + 4 * kh;
    float bv[4];
    unpack4<TB>(braw[j], bv);
    if constexpr (!PRE_D) load_direct(j);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int m = m0 + wm * TM + 16 * i + fr;
      if (n < g.n && m < g.m) {
        float rv[4], a4[4];
        unpack4<TR>(rraw[j][i], rv);
#pragma unroll
        for (int e = 0; e < 4; ++e) a4[e] = acc[j][i][e];
        gemm_finish4<TC, QKV>(g, m, n, a4, bv, rv, QKV || gemm_row_valid(g, m));
      }
    }
  }
}

template <typename T, typename TC, typename TR, bool QKV, int BM, int BN, int NS, bool KS4 = false>
static int launch_cfg(const GemmArgs& g0, hipStream_t st) {
  GemmArgs g = g0;
  auto al = [](const void* p, int bytes) { return ((uintptr_t)p % bytes) == 0; };
  // 16-byte staged epilogue: 16-bit C (and residual), whole 8-column groups;
  // V^T tiles also need whole 16-column blocks of V and at most two sequences
  // per tile.
  g.stage16 = sizeof(TC) == 2 && !(g.epi & TX_EPI_SPLIT_OUT) && g.n % 8 == 0 && g.ldc % 8 == 0 && al(g.c, 16) &&
              (!(g.epi & TX_EPI_RESIDUAL) || (g.ldr % 8 == 0 && al(g.res, 16))) &&
              (!QKV || (g.qk_cols % 16 == 0 && g.seq >= BM && g.ldvt % 8 == 0 && al(g.vt, 16)));
  const long tiles = (long)((g.m + BM - 1) / BM) * ((g.n + BN - 1) / BN);
  if (tiles > 0x7fffffffL) return TX_EUNSUPPORTED;
  gemm_ring_kernel<T, TC, T, TR, BM, BN, NS, QKV, KS4><<<dim3((unsigned)tiles), dim3(512), 0, st>>>(g);
  return hipGetLastError() == hipSuccess ? TX_OK : TX_EHIP;
}

template <typename T, typename TC, typename TR, bool QKV>
static int launch_typed(const GemmArgs& g, int cfg, bool ks4, hipStream_t st) {
  switch (cfg) {
    case 0:
      return ks4 ? launch_cfg<T, TC, TR, QKV, 64, 64, 4, true>(g, st) : launch_cfg<T, TC, TR, QKV, 64, 64, 4>(g, st);
    case 1:
      return ks4 ? launch_cfg<T, TC, TR, QKV, 64, 128, 4, true>(g, st) : launch_cfg<T, TC, TR, QKV, 64, 128, 4>(g, st);
    case 2: return launch_cfg<T, TC, TR, QKV, 128, 128, 4>(g, st);  // 128 KB of LDS
    case 3: return launch_cfg<T, TC, TR, QKV, 128, 128, 2>(g, st);  // 64 KB
    case 4: return launch_cfg<T, TC, TR, QKV, 128, 192, 3>(g, st);  // 120 KB
    case 5: return launch_cfg<T, TC, TR, QKV, 128, 192, 2>(g, st);  // 80 KB
    default: return TX_EUNSUPPORTED;
  }
}

int launch_gemm_ring(const GemmArgs& g, int ab_dt, int c_dt, int res_dt, bool qkv, int cfg, bool ks4,
                     hipStream_t st) {
  if (ab_dt == TX_BF16) {
    if (c_dt == TX_BF16)
      return qkv ? launch_typed<bf16, bf16, bf16, true>(g, cfg, ks4, st)
                 : launch_typed<bf16, bf16, bf16, false>(g, cfg, ks4, st);
    return res_dt == TX_F32 ? launch_typed<bf16, float, float, false>(g, cfg, ks4, st)
                            : launch_typed<bf16, float, bf16, false>(g, cfg, ks4, st);
  }
  if (c_dt == TX_F16)
    return qkv ? launch_typed<f16, f16, f16, true>(g, cfg, ks4, st)
               : launch_typed<f16, f16, f16, false>(g, cfg, ks4, st);
  return res_dt == TX_F32 ? launch_typed<f16, float, float, false>(g, cfg, ks4, st)
                          : launch_typed<f16, float, f16, false>(g, cfg, ks4, st);
}

}  // namespace tx
