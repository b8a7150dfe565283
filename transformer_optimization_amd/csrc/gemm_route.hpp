// Which GEMM kernel a shape takes: the tile configurations of
// gemm_ring_kernel and gemm_hp_kernel and the models of their launch times.
// Plain C++ (no HIP): a test compiles this header with the host compiler and
// checks the choices against measured times.
#pragma once

#include <stdint.h>

namespace tx {

// Tile configurations: BM, BN, workgroups resident per CU (LDS stages in
// launch_typed), and the launch time's model
//   t = c + rounds (a k + e + gelu g),
// rounds of at most `per_cu` tiles a CU; a last round of at most one tile a
// CU runs at its own rate (a1, e1, g / 2).  Least squares over 290 random
// shapes (M 257 .. 20000, N and K the projections and MLPs of d_model 256 ..
// 2048, operands rotated through six sets; standard error 6-10%),
// microseconds.  Picking the least modelled time is 1-3% off the best
// configuration of each shape, and against the 256-row tiles alone 1.65 times
// the speed up to M = 12000 (geometric mean; at M = 1024, N = 512, K = 2048: 28 ->
// 9.4 us) and 1.07 times over M 2600 .. 20000 at d_model 1024 and 2048.
struct GemmRingCfg {
  int bm, bn, per_cu;
  double c, a, e, g, a1, e1;
};
static const GemmRingCfg GEMM_RING[] = {
    {64, 64, 2, 2.76, 0.00568, 1.73, 0.613, 0.00356, 0.965},
    {64, 128, 1, 1.69, 0.00484, 2.54, 1.05, 0.00484, 2.54},
    {128, 128, 1, 0.967, 0.00727, 4.27, 2.16, 0.00727, 4.27},
    {128, 128, 2, 2.48, 0.0144, 3.43, 3.47, 0.0108, 1.82},
    {128, 192, 1, 0.0, 0.00923, 6.13, 3.27, 0.00923, 6.13},
    {128, 192, 2, 2.43, 0.0185, 5.66, 5.3, 0.0121, 2.94},
};

inline double gemm_ring_us(int cfg, int m, int n, int k, bool gelu, int cus) {
  const GemmRingCfg& r = GEMM_RING[cfg];
  const long tiles = (long)((m + r.bm - 1) / r.bm) * ((n + r.bn - 1) / r.bn), slots = (long)cus * r.per_cu;
  const long full = tiles / slots, rem = tiles - full * slots;
  const double g = gelu ? r.g : 0.0;
  double t = r.c + (double)full * (r.a * k + r.e + g);
  if (rem > 0) t += rem <= cus ? r.a1 * k + r.e1 + g / r.per_cu : r.a * k + r.e + g;
  return t;
}

// The configuration of least modelled time for the shape (us in *cost); ks4:
// of those that have the four-sum order.
inline int gemm_ring_pick(int m, int n, int k, bool gelu, int cus, bool ks4, double* cost) {
  int best = 0;
  for (int c = 0; c < (ks4 ? 2 : (int)(sizeof(GEMM_RING) / sizeof(GEMM_RING[0]))); ++c) {
    const double t = gemm_ring_us(c, m, n, k, gelu, cus);
    if (c == 0 || t < *cost) {
      best = c;
      *cost = t;
    }
  }
  return best;
}

// Tile width of gemm_hp_kernel for a shape: the least of
//   w(BN) * BN * (rounds(BN) * K + 1000),
// rounds = ceil(tiles / CUs) (one workgroup per CU), 1000 ~ the exposed last
// epilogue and pipeline fill in units of K, w = 0.97, 1, 1.2 for 256, 192,
// 128 (per-FLOP cost of the narrower wave tiles).  Fitted to every c3/c4
// GEMM shape with all three widths timed in one process and checked on
// whole forwards: it picks 256 for c3's FFN-in and c4's out_proj, FFN-in and
// FFN-out, 128 for c3's out_proj and FFN-out.  (192 for the c3 and c4 QKV
// projections, which take 128 x 192 ring tiles now; at c4's the 256-wide tiles won
// in isolation, 172 vs 181 us, but not inside the forward, where their two K
// stages see cold operands.)  gemm_hp_us below does not always agree with it:
// 4096x4096x1024 with GELU is 128 here and modelled 40.6 us at 256 against 46.0
// at 128; which is right has not been measured.
inline int gemm_hp_width(int m, int n, int k, int cus) {
  static const int bn[3] = {256, 192, 128};
  static const double w[3] = {0.97, 1.0, 1.2};
  int best = 256;
  double best_cost = 0.0;
  for (int c = 0; c < 3; ++c) {
    const long tiles = (long)((m + 255) / 256) * ((n + bn[c] - 1) / bn[c]);
    const long rounds = (tiles + cus - 1) / cus;
    const double cost = w[c] * bn[c] * ((double)rounds * k + 1000.0);
    if (c == 0 || cost < best_cost) {
      best = bn[c];
      best_cost = cost;
    }
  }
  return best;
}

// Modelled time (us) of gemm_hp_kernel at a tile width: c + rounds (a k + e +
// gelu g), fitted to the same random shapes as gemm_ring_kernel's
// configurations (standard error 8-9%).
inline double gemm_hp_us(int bn, int m, int n, int k, bool gelu, int cus) {
  const int i = bn == 256 ? 0 : bn == 192 ? 1 : 2;
  static const double c[3] = {0.0, 0.0402, 0.666}, a[3] = {0.0224, 0.018, 0.0123}, e[3] = {10.1, 8.55, 6.29},
                      g[3] = {7.59, 5.17, 3.77};
  const long tiles = (long)((m + 255) / 256) * ((n + bn - 1) / bn);
  const long rounds = (tiles + cus - 1) / cus;
  return c[i] + (double)rounds * (a[i] * k + e[i] + (gelu ? g[i] : 0.0));
}

// What the choice among the kernels of M >= 256 looks at.
struct GemmShape {
  int m, n, k;
  bool gelu, residual;
  bool f32;    // fp32 C, one value per element
  bool split;  // hi / lo pairs
  bool qkv;
  int seq;     // qkv
};

// The kernel of a shape with M >= 256: 1000 + i = gemm_ring_kernel's
// configuration i, 256 / 192 / 128 = gemm_hp_kernel at that width, 20 =
// gemm_big_kernel.  ring_ok: gemm_ring_kernel takes the operands.
inline int gemm_route(const GemmShape& s, int cus, bool ring_ok) {
  // gemm_hp_kernel writes V^T element by element when a 16-row chunk can span
  // two sequences; gemm_ring_kernel does not.  Sequences of 421 to 1645 against
  // ones of whole 16 rows and nearly the same length, d_model 512, 1024, 2048: the
  // 256-row tiles take 1.08 to 1.8 times as long, ring tiles 1.04 to 1.4
  // (2105x3072x1024 24.4 us on 128-wide tiles and 21.9 on ring tiles, modelled
  // 19.6 and 20.7).  With 1.2 eight of the nine are within 2% of their best kernel;
  // 2105x6144x2048 takes 78 us on 256-wide tiles, 63 on ring tiles.
  const double ragged = s.qkv && s.seq % 16 != 0 ? 1.2 : 1.0;
  // Tall operands (A streams from HBM rather than staying in the caches) with a
  // short K panel: of the 256-row tiles the 128-wide ones, whose third K stage
  // covers the longer latency.  The fit ends at 20000 rows; here, relative to
  // the 256-row tiles, the 128 x 128 ring tiles take longer than modelled except
  // beside a GELU and for pairs, and the 128 x 192 ones where the epilogue writes
  // four bytes an element without reading a residual.  The factors come from 321
  // random calls with M 32768 .. 131072: 0.947 of the time of the 256-row tiles
  // alone (geometric mean; 7 calls over 1.03, the longest 1.06), without them
  // 0.954 (42 calls over 1.03, the longest 1.12).  In us, 256-row / 128x128 /
  // 128x192: fp32 35138x768x768 75 / 75 / 84, fp32 121852x1024x1024 368 / 398 / 370,
  // pairs 107795x2048x512 533 / 500 / 580, 16-bit 130663x1024x1024 345 / 363 / 342.
  if (s.m >= 32768 && s.k <= 2048) {
    const double hp = gemm_hp_us(128, s.m, s.n, s.k, s.gelu, cus) * ragged;
    const double r128 = gemm_ring_us(3, s.m, s.n, s.k, s.gelu, cus) * (s.split ? 0.95 : s.gelu ? 1.0 : 1.15);
    const double r192 = gemm_ring_us(5, s.m, s.n, s.k, s.gelu, cus) * (s.gelu || s.qkv ? 1.0 : 1.03);
    const bool no192 = s.split || (s.f32 && !s.residual);
    if (!ring_ok || hp <= (no192 || r128 < r192 ? r128 : r192)) return 128;
    return no192 || r128 < r192 ? 1003 : 1005;
  }
  double ring = 0.0;
  const int cfg = gemm_ring_pick(s.m, s.n, s.k, s.gelu, cus, false, &ring);
  // fp32 C with short K: gemm_hp_kernel's staged epilogue covers 16-bit C only,
  // and its direct fp32 epilogue lost to the 128x128 kernel; ring tiles are
  // faster than that one everywhere (16000x1024x1024 53 to 55 against 56 us,
  // 5003x1024x1024 20 against 26 us, 98477x2048x3072 1367 against 1621).
  if (s.f32 && s.k < 4096) return ring_ok ? 1000 + cfg : 20;
  // Smaller tiles where their modelled time is less.
  const int bn = gemm_hp_width(s.m, s.n, s.k, cus);
  return ring_ok && ring < gemm_hp_us(bn, s.m, s.n, s.k, s.gelu, cus) * ragged ? 1000 + cfg : bn;
}

}  // namespace tx
