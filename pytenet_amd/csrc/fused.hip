// H_eff and environment steps of small bonds in one launch.
//
// The three contractions (ops.hip) are product - MPO mode mix - product, of which the last
// sums over one bond and leaves the other free: for a range of the free bond's index (r' of
// H_eff, rb of the left and l of the right environment step) the whole chain depends on
// nothing outside it. A workgroup takes such a range and keeps T1 and T2 of it in LDS.
//   by columns (H_eff, left step):  T1[(x, i1), (j1, y)] = sum_k A[(x, i1), k] B[k, (j1, y)],
//     T2 = mix(T1), out[u, (j2, y)] = sum_(x, i2) F[(x, i2), u] T2[(x, i2), (j2, y)], y in a range
//   by rows (right step): the same T1 and T2 for x in a range,
//     out[(x, i2), u] = sum_(j2, y) T2[(x, i2), (j2, y)] conj(F[u, (j2, y)])
// As three launches these are bound by the launches and by the latency of a few dependent steps
// each (3.3 - 7 us); here by the products of one CU, so the form pays up to about 9500 estimated
// matrix cycles. Calls of the library in a loop, three launches against one: left step D = 8
// 15.4 -> 10.9 us, 24 15.2 -> 10.3, 32 15.0 -> 12.0 (8200 cycles), 48 14.8 -> 19.6 (18000); right step
// 24 14.8 -> 12.8 (9200); H_eff of one site D = 24 20.0 -> 9.9, of two 14.4 -> 10.9.
#include <algorithm>
#include <cmath>
#include "ops.h"
#include "wave.h"
#include "wave_product.h"

namespace ptn {

constexpr int FU_T = 512;
constexpr int FU_LDS = 136 * 1024;
constexpr int FU_MIX = 32;                // largest row or column count of the MPO matrix
constexpr double FU_CYCLES = 9500.0;      // limit of the estimate in fused_plan

struct FusedArgs {
  int rows;                               // range over x instead of y
  int X, Y, range, i1, j1, i2, j2, wtrans;
  int ld1, ld2, o_t2, o_mpo, parts;
  float ry;                               // 1 / (columns of the range): exact quotients below 2^14
  SmallProduct g1, g3;
  const double2 *a, *b, *w, *f;
  double2* out;
  int64_t sa, sb, sw, sf, so;             // strides of a batch
  const int* skip;
  int64_t skip_stride;
};

template <bool ROWS, bool CONJ1>
__global__ __launch_bounds__(FU_T) void k_fused_apply(FusedArgs g) {
  __shared__ __align__(16) double2 lds[FU_LDS / 16];
  __shared__ int part_end[FU_MIX + 1], used[FU_MIX], count[FU_MIX * FU_MIX / 64];
  __shared__ short src[FU_MIX * FU_MIX], dst[FU_MIX * FU_MIX], row[FU_MIX * FU_MIX];
  if (g.skip && g.skip[blockIdx.y * g.skip_stride]) return;
  const int t = threadIdx.x, z = blockIdx.y, r0 = blockIdx.x * g.range;
  const double2* A = g.a + z * g.sa + (ROWS ? (int64_t)r0 * g.i1 * g.g1.am : 0);
  const double2* B = g.b + z * g.sb;
  const double2* F = g.f + z * g.sf;
  double2* out = g.out + z * g.so;
  double2 *t1 = lds, *t2 = lds + g.o_t2, *mpo = lds + g.o_mpo;
  // x and y of this workgroup: rows nx, columns ny of T1 per (i1, j1)
  const int nx = ROWS ? min(g.range, g.X - r0) : g.X;
  const int ny = ROWS ? g.Y : g.range, ylast = g.Y - 1;
  const int ni = g.i1 * g.j1, no = g.i2 * g.j2;

  // the MPO matrix's nonzero entries in the order of (output, input)
  double2 we[2];
  unsigned long long has[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int e = t + c * FU_T, o = e / ni, i = e - o * ni;
    we[c] = e < no * ni ? g.w[z * g.sw + (g.wtrans ? i * no + o : e)] : make_double2(0.0, 0.0);
    has[c] = __ballot(we[c].x != 0.0 || we[c].y != 0.0);
    if ((t & 63) == 0) count[c * (FU_T / 64) + (t >> 6)] = __popcll(has[c]);
  }
  if (t < no) used[t] = 0;
  // first product
  {
    SmallProduct p = g.g1;
    if (ROWS && nx < g.range) p.M = nx * g.i1;
    small_product<CONJ1>(
        p, A, B,
        [&](int n) {
          const int j = (int)(((float)n + 0.5f) * g.ry), y = n - j * ny;
          return j * g.Y + (ROWS ? y : min(r0 + y, ylast));
        },
        [&](int, int m, int n, int part) { return (double*)&t1[m * g.ld1 + n] + part; });
  }
  __syncthreads();
  {
    int at = 0, total = 0;
    constexpr int NC = 2 * FU_T / 64;
    int before[2] = {0, 0};
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      const int n = count[q];
#pragma unroll
      for (int c = 0; c < 2; ++c) before[c] += q < c * (FU_T / 64) + (t >> 6) ? n : 0;
      total += n;
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
      if (has[c] >> (t & 63) & 1) {
        at = before[c] + __popcll(has[c] & ((1ull << (t & 63)) - 1));
        const int e = t + c * FU_T, o = e / ni, i = e - o * ni;
        mpo[at] = we[c];
        src[at] = (short)(i / g.j1 * g.ld1 + i % g.j1 * ny);
        row[at] = (short)o;
        used[o] = 1;
      }
    __syncthreads();
    // a row's last entry stores it; a row without entries is zero
    for (int c = t; c < total; c += FU_T) {
      const int o = row[c];
      dst[c] = c + 1 == total || row[c + 1] != o ? (short)(o / g.j2 * g.ld2 + o % g.j2 * ny)
                                                 : (short)-1;
    }
    if (t < no && !used[t])
      for (int x = 0; x < nx; ++x)
        for (int y = 0; y < ny; ++y)
          t2[(x * g.i2 + t / g.j2) * g.ld2 + t % g.j2 * ny + y] = make_double2(0.0, 0.0);
    if (t <= g.parts) {   // parts of whole rows with about the same number of entries
      int c = total * t / g.parts;
      while (c > 0 && c < total && row[c] == row[c - 1]) ++c;
      part_end[t] = c;
    }
  }
  __syncthreads();
  {
    // a thread takes a unit (x, y) and a part of the rows' entries
    const int units = nx * ny, per = FU_T / g.parts;
    const int part = __builtin_amdgcn_readfirstlane(t / per);
    if (part < g.parts) {
      const int e0 = part_end[part], e1 = part_end[part + 1];
      for (int u = t - part * per; u < units; u += per) {
        const int x = (int)(((float)u + 0.5f) * g.ry), y = u - x * ny;
        const double2* in = t1 + x * g.i1 * g.ld1 + y;
        double2* to = t2 + x * g.i2 * g.ld2 + y;
        double yr = 0.0, yi = 0.0;
        for (int e = e0; e < e1; e += 4) {
          double2 c[4], v[4];
          int at[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int f = min(e + q, e1 - 1);
            c[q] = mpo[f];
            at[q] = dst[f];
            v[q] = in[src[f]];
          }
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (e + q < e1) {
              yr = fma(c[q].x, v[q].x, fma(-c[q].y, v[q].y, yr));
              yi = fma(c[q].x, v[q].y, fma(c[q].y, v[q].x, yi));
              if (at[q] >= 0) {
                to[at[q]] = make_double2(yr, yi);
                yr = yi = 0.0;
              }
            }
        }
      }
    }
  }
  __syncthreads();
  if (ROWS) {
    SmallProduct p = g.g3;
    if (nx < g.range) p.M = nx * g.i2;
    const int64_t ldf = (int64_t)g.j2 * g.Y, U = p.N;
    double2* o = out + (int64_t)r0 * g.i2 * U;
    if (p.ks == 1) {
      small_product<true>(p, (const double2*)t2, F, [&](int n) { return n * ldf; },
                          [&](int, int m, int n, int part) { return (double*)&o[m * U + n] + part; });
      return;
    }
    const int size = p.M * p.N;
    small_product<true>(p, (const double2*)t2, F, [&](int n) { return n * ldf; },
                        [&](int q, int m, int n, int part) {
                          return (double*)&t1[q * size + m * (int)U + n] + part;
                        });
    __syncthreads();
    for (int e = t; e < size; e += FU_T) {
      double2 v = t1[e];
      for (int q = 1; q < p.ks; ++q) {
        v.x += t1[q * size + e].x;
        v.y += t1[q * size + e].y;
      }
      o[e] = v;
    }
  } else {
    const SmallProduct& p = g.g3;
    const int64_t ldo = (int64_t)g.j2 * g.Y;
    const auto same = [](int n) { return n; };
    const int size = p.M * p.N;
    small_product<false>(p, F, (const double2*)t2, same, [&](int q, int m, int n, int part) {
      return (double*)&t1[q * size + m * p.N + n] + part;
    });
    __syncthreads();
    const float rn = 1.0f / (float)p.N;
    for (int e = t; e < size; e += FU_T) {
      const int m = (int)(((float)e + 0.5f) * rn), n = e - m * p.N;
      const int j = (int)(((float)n + 0.5f) * g.ry), y = n - j * ny;
      double2 v = t1[e];
      for (int q = 1; q < p.ks; ++q) {
        v.x += t1[q * size + e].x;
        v.y += t1[q * size + e].y;
      }
      if (r0 + y < g.Y) out[m * ldo + (int64_t)j * g.Y + r0 + y] = v;
    }
  }
}

// Layout of a contraction for the one-launch form; false if it does not fit or if the
// products of one workgroup are estimated above FU_CYCLES (matrix cycles of one SIMD with
// its tiles rounded up to the waves).
static bool fused_plan(bool rows, int64_t X, int64_t Y, int64_t K, int64_t U, int i1, int j1, int i2,
                       int j2, FusedArgs* g) {
  if (X < 1 || Y < 1 || K < 1 || U < 1 || X > 1024 || Y > 1024 || K > 1024 || U > 1024) return false;
  if (i1 * j1 > FU_MIX || i2 * j2 > FU_MIX) return false;
  auto pad = [](int64_t n) { return n % 16 ? n : n + 8; };   // rows half a turn of the banks apart
  // the range: at least 8 columns (or 16 rows) in both products
  const int64_t least = rows ? (16 + std::min(i1, i2) - 1) / std::min(i1, i2)
                             : (8 + std::min(j1, j2) - 1) / std::min(j1, j2);
  const int64_t range = std::min<int64_t>(least, rows ? X : Y);
  const int64_t nx = rows ? range : X, ny = rows ? Y : range;
  const int64_t n1 = j1 * ny, n2 = j2 * ny;
  g->rows = rows;
  g->X = (int)X;
  g->Y = (int)Y;
  g->range = (int)range;
  g->i1 = i1;
  g->j1 = j1;
  g->i2 = i2;
  g->j2 = j2;
  g->ld1 = (int)pad(n1);
  g->ld2 = (int)pad(n2);
  const int64_t s1 = nx * i1 * g->ld1, s2 = nx * i2 * g->ld2;
  const int64_t M3 = rows ? nx * i2 : U, N3 = rows ? U : n2, K3 = rows ? n2 : nx * i2;
  // parts of k in the last product while half of the waves would be idle; they lie over T1
  const int64_t tiles = (M3 + 15) / 16 * ((N3 + 7) / 8), steps = (K3 + 3) / 4;
  int ks = 1;
  while (ks < 8 && tiles * ks * 2 <= FU_T / 64 && steps >= 4 * ks) ks *= 2;
  const int64_t t1 = std::max(s1, rows && ks == 1 ? 0 : ks * M3 * N3);
  g->o_t2 = (int)t1;
  g->o_mpo = (int)(t1 + s2);
  if ((t1 + s2 + (int64_t)i1 * j1 * i2 * j2) * 16 > FU_LDS) return false;
  if (t1 >= 16384 || s2 >= 16384) return false;
  g->g1 = small_product_of(nx * i1, n1, K, K, 1, (int64_t)j1 * Y, 1);
  if (rows) g->g3 = small_product_of(M3, N3, K3, g->ld2, 1, 1, ks);
  else g->g3 = small_product_of(M3, N3, K3, 1, U, g->ld2, ks);
  const double w = FU_T / 64, simd = 4;
  const double c1 = std::ceil(g->g1.tiles / w) * (w / simd) * ((K + 3) / 4) * 128.0;
  const double c3 = std::ceil(g->g3.tiles / w) * (w / simd) * g->g3.per * 128.0;
  if (c1 + c3 > FU_CYCLES) return false;
  g->ry = 1.0f / (float)ny;
  const int64_t units = (nx * ny + 63) / 64 * 64;
  int64_t parts = std::max<int64_t>(1, std::min<int64_t>(FU_T / units, i2 * j2));
  while (FU_T % parts || (FU_T / parts) % 64) --parts;
  g->parts = (int)parts;
  return true;
}

// Runs the contraction of `kind` in one launch if that applies (FP64, dense, complex128
// operands, an output apart from everything that is read); operands as in heff_apply,
// env_left and env_right (f: L, A or B). Sets done.
int fused_apply(int kind, const Dims& D, const void* a, const void* b, const void* w, const void* f,
                void* out, hipStream_t s, int64_t batch, bool* done) {
  *done = false;
  if (batch > 65535) return PTN_OK;
  FusedArgs g{};
  const int d = (int)D.d, Ml = (int)D.Ml, Mr = (int)D.Mr;
  if (D.d > FU_MIX || D.Ml > FU_MIX || D.Mr > FU_MIX) return PTN_OK;
  const int64_t nA = D.Dl * D.d * D.Dr, nL = D.Dl * D.Ml * D.Dl, nR = D.Dr * D.Mr * D.Dr;
  bool ok;
  if (kind == FUSED_HEFF) {
    ok = fused_plan(false, D.Dl, D.Dr, D.Dr, D.Dl, d, Mr, Ml, d, &g);
    g.sa = nA; g.sb = nR; g.sf = nL; g.so = nA;
  } else if (kind == FUSED_ENV_LEFT) {
    ok = fused_plan(false, D.Dl, D.Dr, D.Dl, D.Dr, Ml, d, d, Mr, &g);
    g.wtrans = 1;
    g.sa = nL; g.sb = nA; g.sf = nA; g.so = nR;
  } else {
    ok = fused_plan(true, D.Dl, D.Dr, D.Dr, D.Dl, d, Mr, Ml, d, &g);
    g.sa = nA; g.sb = nR; g.sf = nA; g.so = nL;
  }
  if (!ok) return PTN_OK;
  g.sw = D.Ml * D.d * D.d * D.Mr;
  auto apart = [&](const void* p, int64_t n) {
    const char *o = (const char*)out, *x = (const char*)p;
    return x + batch * n * 16 <= o || o + batch * g.so * 16 <= x;
  };
  if (!apart(a, g.sa) || !apart(b, g.sb) || !apart(f, g.sf) || !apart(w, g.sw)) return PTN_OK;
  g.a = (const double2*)a;
  g.b = (const double2*)b;
  g.w = (const double2*)w;
  g.f = (const double2*)f;
  g.out = (double2*)out;
  g.skip = skip_flag().p;
  g.skip_stride = skip_flag().stride;
  const int64_t free_len = g.rows ? D.Dl : D.Dr;
  const dim3 grid((unsigned)((free_len + g.range - 1) / g.range), (unsigned)batch);
  const double flop = 8.0 * (double)batch *
                      ((double)g.X * g.i1 * g.j1 * g.Y * g.g1.K +
                       (g.rows ? (double)g.X * g.i2 * g.g3.N * g.g3.K
                               : (double)g.g3.M * g.j2 * g.Y * g.g3.K));
  const double bytes = 16.0 * (double)batch * (double)(g.sa + g.sb + g.sw + g.sf + g.so);
  if (kind == FUSED_HEFF)
    tlaunch("k_fused_apply<heff>", flop, bytes, k_fused_apply<false, false>, grid, dim3(FU_T), s, g);
  else if (kind == FUSED_ENV_LEFT)
    tlaunch("k_fused_apply<left>", flop, bytes, k_fused_apply<false, true>, grid, dim3(FU_T), s, g);
  else
    tlaunch("k_fused_apply<right>", flop, bytes, k_fused_apply<true, false>, grid, dim3(FU_T), s, g);
  PTN_LAUNCH_CHECK();
  *done = true;
  return PTN_OK;
}

}  // namespace ptn
