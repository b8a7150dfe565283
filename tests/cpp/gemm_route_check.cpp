// The kernel choice of csrc/gemm_route.hpp against measured times (us, one
// MI355X of 256 CUs, the three kernels in turn): tall calls where the 256-row
// kernel, the 128 x 128 or the 128 x 192 ring tiles differ.  The chosen one may
// take at most 1.04 times the 256-row kernel's time and 1.10 times the least
// (two runs of one kernel differ by up to 3%).  Prints "ok" or what failed.
#include <stdio.h>

#include "gemm_route.hpp"

enum { PLAIN, GELU, RES, F32, F32RES, SPLIT, QKV };
struct Call {
  int kind, m, n, k, seq;
  double hp, r128, r192;
};
static const Call CALLS[] = {
    {F32, 35138, 768, 768, 0, 74.8, 75.4, 83.8},      {F32, 77845, 768, 768, 0, 163.3, 161.7, 176.3},
    {F32, 104912, 1024, 1024, 0, 320.2, 342.2, 316.4}, {F32, 121852, 1024, 1024, 0, 367.7, 398.3, 370.0},
    {F32, 60425, 512, 512, 0, 75.4, 79.7, 74.0},       {F32, 46010, 256, 256, 0, 21.7, 18.1, 23.2},
    {F32, 35452, 512, 512, 0, 38.2, 32.7, 33.7},       {F32RES, 121646, 1024, 1024, 0, 435.1, 455.6, 441.8},
    {F32RES, 37159, 256, 256, 0, 31.9, 24.4, 26.7},    {RES, 130663, 1024, 1024, 0, 345.1, 363.2, 341.6},
    {RES, 67995, 1024, 1024, 0, 182.4, 193.8, 177.4},  {RES, 72305, 256, 256, 0, 31.4, 25.2, 29.9},
    {PLAIN, 110319, 512, 512, 0, 87.9, 94.1, 85.4},    {PLAIN, 120960, 1024, 1024, 0, 281.1, 301.1, 282.5},
    {PLAIN, 34499, 768, 768, 0, 60.8, 56.6, 51.5},     {PLAIN, 39895, 256, 256, 0, 18.0, 14.0, 17.1},
    {SPLIT, 107795, 2048, 512, 0, 532.8, 500.4, 579.5}, {SPLIT, 43232, 1536, 768, 0, 215.0, 198.4, 230.4},
    {GELU, 41364, 2048, 1024, 0, 247.9, 226.7, 206.9}, {GELU, 36758, 512, 256, 0, 32.3, 24.2, 25.9},
    {QKV, 66560, 3072, 1024, 65, 477.0, 480.0, 447.4}, {QKV, 55296, 1536, 512, 768, 125.7, 113.8, 115.5},
};

int main() {
  int fails = 0;
  for (const Call& c : CALLS) {
    tx::GemmShape s{};
    s.m = c.m;
    s.n = c.n;
    s.k = c.k;
    s.gelu = c.kind == GELU || c.kind == SPLIT;
    s.residual = c.kind == RES || c.kind == F32RES;
    s.f32 = c.kind == F32 || c.kind == F32RES;
    s.split = c.kind == SPLIT;
    s.qkv = c.kind == QKV;
    s.seq = c.seq;
    const int v = tx::gemm_route(s, 256, true);
    const double t = v == 128 ? c.hp : v == 1003 ? c.r128 : v == 1005 ? c.r192 : 1e9;
    double least = c.hp < c.r128 ? c.hp : c.r128;
    if (c.r192 < least) least = c.r192;
    if (t > 1.04 * c.hp || t > 1.10 * least) {
      printf("FAIL kind %d %dx%dx%d: kernel %d, %.1f us against %.1f / %.1f / %.1f\n", c.kind, c.m, c.n, c.k, v, t,
             c.hp, c.r128, c.r192);
      ++fails;
    }
    if (tx::gemm_route(s, 256, false) >= 1000) {
      printf("FAIL %dx%dx%d: ring tiles for operands they do not take\n", c.m, c.n, c.k);
      ++fails;
    }
  }
  if (!fails) printf("ok\n");
  return fails != 0;
}
