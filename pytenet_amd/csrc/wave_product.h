// Complex FP64 products of a few thousand outputs inside one workgroup, for kernels that
// chain several of them.
#pragma once
#include "common.h"

namespace ptn {

// C = A . B (B conjugated with CONJ) with M x N outputs and K terms in ks parts, by the
// waves of one workgroup: A(m, k) at a[m * am + k * ak], B(k, n) at b[k * bk + bcol(n)]; the
// real (part 0) or imaginary part of part p of output (m, n) goes to st(p, m, n, part). A wave
// takes tiles of 16 x 8 (tn of them per row of tiles, tk = tn ks with the parts); rows and
// columns beyond the ends repeat the last ones, terms beyond K are zero.
struct SmallProduct {
  int M, N, K, am, ak, bk, ks, per, tk, tn, tiles;
  float rk, rn;                           // 1 / tk, 1 / tn: exact quotients below 2^14
};
inline SmallProduct small_product_of(int64_t M, int64_t N, int64_t K, int64_t am, int64_t ak,
                                     int64_t bk, int ks) {
  SmallProduct p{};
  p.M = (int)M;
  p.N = (int)N;
  p.K = (int)K;
  p.am = (int)am;
  p.ak = (int)ak;
  p.bk = (int)bk;
  p.ks = ks;
  p.per = (int)((K + 4 * ks - 1) / (4 * ks));
  p.tn = (int)((N + 7) / 8);
  p.tk = p.tn * ks;
  p.tiles = (int)((M + 15) / 16) * p.tk;
  p.rk = 1.0f / (float)p.tk;
  p.rn = 1.0f / (float)p.tn;
  return p;
}
template <bool CONJ, typename PA, typename PB, typename FC, typename FS>
__device__ __forceinline__ void small_product(const SmallProduct& g, PA a, PB b, FC bcol, FS st) {
  constexpr int U = 2;                    // steps per batch of loads
  const int lane = threadIdx.x & 63, l16 = lane & 15, kk = lane >> 4, pb = lane & 1;
  const int nw = blockDim.x >> 6, whole = g.K >> 2;
  for (int t = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); t < g.tiles; t += nw) {
    const int mt = __builtin_amdgcn_readfirstlane((int)(((float)t + 0.5f) * g.rk));
    const int q = t - mt * g.tk;
    const int p = __builtin_amdgcn_readfirstlane((int)(((float)q + 0.5f) * g.rn));
    const int m0 = 16 * mt, n0 = 8 * (q - p * g.tn);
    const int s0 = p * g.per, s1 = min(s0 + g.per, whole);   // whole steps of four k
    const int col = n0 + (l16 >> 1);
    const PA ra = a + min(m0 + l16, g.M - 1) * g.am + kk * g.ak;
    const PB rb = b + bcol(min(col, g.N - 1)) + kk * g.bk;
    d4_t acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
    double2 xa[U], xb[U], ya[U], yb[U];
    auto load = [&](int s, double2 (&fa)[U], double2 (&fb)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (s + u < s1) {
          fa[u] = ra[4 * (s + u) * g.ak];
          fb[u] = rb[4 * (s + u) * g.bk];
        }
    };
    auto step = [&](double2 fa, double2 fb) {
      if (CONJ) fb.y = -fb.y;
      acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(fa.x, pb ? fb.y : fb.x, acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(fa.y, pb ? fb.x : -fb.y, acc1, 0, 0, 0);
    };
    auto multiply = [&](int s, const double2 (&fa)[U], const double2 (&fb)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (s + u < s1) step(fa[u], fb[u]);
    };
    load(s0, xa, xb);
    for (int s = s0; s < s1; s += 2 * U) {
      load(s + U, ya, yb);
      multiply(s, xa, xb);
      load(s + 2 * U, xa, xb);
      multiply(s + U, ya, yb);
    }
    if ((g.K & 3) && p == g.ks - 1) {     // the last terms
      const bool in = 4 * whole + kk < g.K;
      const double2 z = make_double2(0.0, 0.0);
      step(in ? ra[4 * whole * g.ak] : z, in ? rb[4 * whole * g.bk] : z);
    }
    // result element v: row lane / 16 + 4 v, column lane % 16 (real and imaginary parts)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = m0 + kk + 4 * v;
      if (row < g.M && col < g.N) *st(p, row, col, pb) = acc0[v] + acc1[v];
    }
  }
}

}  // namespace ptn
