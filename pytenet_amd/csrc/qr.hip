// Householder QR of a complex128 matrix with LAPACK's conventions, so that Q
// and R agree with numpy.linalg.qr (zgeqrf + zungqr) to rounding, including
// the completion of Q for rank-deficient inputs:
//   reflector j from alpha = A[j, j], x = A[j+1:, j]:
//     xnorm = |x|; if xnorm == 0 and Im(alpha) == 0: tau = 0 (H = I)
//     else beta = -sign(Re alpha) |(alpha, x)|, tau = (beta - alpha) / beta,
//          v = [1, x / (alpha - beta)], R[j, j] = beta (real)
//   A <- H^H A with H = I - tau v v^H;   Q = H_0 H_1 ... H_{k-1} [I_k; 0].
//
// Blocked right-looking algorithm on a column-major copy (panels of QR_NB
// columns):
//   panel:    up to 256 rows one workgroup with the panel in its registers
//             (k_qr_panel); up to 2048 rows one launch for every four columns
//             (k_qr_col4) and above for every two (k_qr_col2r, k_qr_col2; k_qr_col
//             for a last odd column): every workgroup computes the launch's
//             reflectors (the same deterministic reductions) and applies them to
//             one remaining column of the panel;
//   WY form:  T from V^H V (k_qr_vtv, k_qr_tmat), H_j0 ... = I - V T V^H;
//   trailing: A <- A - V (T^H (V^H A)): V^H A as a split-K complex product on
//             MFMA, the sum of the K chunks and the small T^H product in
//             k_qr_reduce, and one accumulating MFMA product.
// Q (or Q times a given matrix) is formed panel by panel in reverse order
// with the same three steps and T in place of T^H.
#include <float.h>
#include "qr.h"
#include "wave.h"

namespace ptn {

// Eight sums over the wave at once: two values fold into one register per step (the
// halves of the wave, then the rows of 16, then of 8 lanes keep one each and add the
// other's partner), so the eight cost little more than one. Lane group g = lane / 8
// ends with the sum of value sum8_slot(g).
__device__ __forceinline__ int sum8_slot(int g) { return (g >> 2) | (g & 2) | ((g & 1) << 2); }
template <bool HALF> __device__ __forceinline__ double swap_add(double a, double b) {
  typedef unsigned int u2 __attribute__((ext_vector_type(2)));
  const unsigned long long x = (unsigned long long)__double_as_longlong(a),
                           y = (unsigned long long)__double_as_longlong(b);
  u2 lo, hi;
  if constexpr (HALF) {
    lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  } else {
    lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  }
  const double p = __longlong_as_double(((long long)hi[0] << 32) | lo[0]);
  const double q = __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
  return p + q;
}
__device__ __forceinline__ double wave_sum8(const double (&v)[8]) {
  double a[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) a[k] = swap_add<true>(v[2 * k], v[2 * k + 1]);
  const double b0 = swap_add<false>(a[0], a[1]), b1 = swap_add<false>(a[2], a[3]);
  const bool upper = (threadIdx.x & 8) != 0;
  double c = upper ? b1 : b0;
  const double d = upper ? b0 : b1;
  c += dpp_rot<0x128>(d);   // row rotate right by 8
  c += dpp_rot<0xB1>(c);    // quad: lanes 1 0 3 2
  c += dpp_rot<0x4E>(c);    // quad: lanes 2 3 0 1
  c += dpp_rot<0x141>(c);   // half-row mirror: the other quad
  return c;
}

// sums of a and b over a 256-thread workgroup, returned to every thread; the
// order of the additions is fixed, so every workgroup that reduces the same
// data gets bitwise the same result
__device__ void block_sum2(double& a, double& b) {
  __shared__ double red[2][4];
  a = wave_sum(a);
  b = wave_sum(b);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { red[0][w] = a; red[1][w] = b; }
  __syncthreads();
  a = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
  b = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
  __syncthreads();
}

// sums of N values over a 256-thread workgroup (fixed order, as block_sum2)
template <int N> __device__ void block_sum(double (&v)[N]) {
  __shared__ double red[N][4];
  const int w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    v[k] = wave_sum(v[k]);
    if ((threadIdx.x & 63) == 0) red[k][w] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = (red[k][0] + red[k][1]) + (red[k][2] + red[k][3]);
  __syncthreads();
}

// Householder reflector from alpha and |x| (LAPACK zlarfg conventions):
// H = I when x = 0 and alpha is real (tau = 0, R entry alpha, v = e_j);
// else beta = -sign(Re alpha) |(alpha, x)|, tau = (beta - alpha) / beta and
// v = [1, x / (alpha - beta)], held as the complex factor sc = 1 / (alpha - beta)
struct Refl {
  double2 tau, rd, sc;
};
__device__ __forceinline__ Refl make_refl(double2 alpha, double xnorm) {
  Refl h;
  if (xnorm == 0.0 && alpha.y == 0.0) {
    h.tau = make_double2(0.0, 0.0);
    h.rd = alpha;
    h.sc = make_double2(0.0, 0.0);
    return h;
  }
  const double ar = fabs(alpha.x), ai = fabs(alpha.y);
  const double mx = fmax(fmax(ar, ai), xnorm);
  const double nrm = mx * sqrt((ar / mx) * (ar / mx) + (ai / mx) * (ai / mx) +
                               (xnorm / mx) * (xnorm / mx));
  const double beta = -copysign(nrm, alpha.x);
  const double dr = alpha.x - beta, di = alpha.y;
  const double den = dr * dr + di * di;
  h.sc = make_double2(dr / den, -di / den);
  h.tau = make_double2((beta - alpha.x) / beta, -alpha.y / beta);
  h.rd = make_double2(beta, 0.0);
  return h;
}
// 1 / x to full precision from the hardware's estimate (normal x)
__device__ __forceinline__ double rcp_full(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(y, fma(-x, y, 1.0), y);
  return fma(y, fma(-x, y, 1.0), y);
}
// the same reflector from the sum of squares s2 = |x|^2, with the short chain of
// operations that the panel kernels wait for; norms far outside the usual range
// take the scaled form
__device__ __forceinline__ Refl make_refl2(double2 alpha, double s2) {
  const double n2 = fma(alpha.x, alpha.x, fma(alpha.y, alpha.y, s2));
  if (!(n2 > 0x1p-900 && n2 < 0x1p900)) return make_refl(alpha, sqrt(s2));
  Refl h;
  if (s2 == 0.0 && alpha.y == 0.0) {
    h.tau = make_double2(0.0, 0.0);
    h.rd = alpha;
    h.sc = make_double2(0.0, 0.0);
    return h;
  }
  const double y = rsq_full(n2);
  double nrm = n2 * y;
  nrm = fma(0.5 * y, fma(-nrm, nrm, n2), nrm);
  const double beta = -copysign(nrm, alpha.x);
  const double dr = alpha.x - beta, di = alpha.y;
  const double iden = rcp_full(fma(dr, dr, di * di)), ib = rcp_full(beta);
  h.sc = make_double2(dr * iden, -di * iden);
  h.tau = make_double2(-dr * ib, -di * ib);
  h.rd = make_double2(beta, 0.0);
  return h;
}
__device__ __forceinline__ double2 cmul2(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 conj2(double2 a) { return make_double2(a.x, -a.y); }

__global__ void k_zero_u64(int64_t n, unsigned long long* __restrict__ p) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0ull;
}

// mxb[b] = largest |Re|, |Im| of matrix b (m x n, lda, at a + b sa): the bit
// patterns of non-negative doubles order like the doubles, so an integer
// atomic max (one per workgroup) gives the float max (NaN entries are skipped
// by fmax)
__global__ __launch_bounds__(256) void k_maxabs(int64_t m, int64_t n, const double2* __restrict__ a,
                                                int64_t lda, int64_t sa,
                                                unsigned long long* __restrict__ mxb) {
  a += blockIdx.y * sa;
  double v = 0.0;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < m * n;
       t += (int64_t)gridDim.x * blockDim.x) {
    const double2 x = a[(t / n) * lda + t % n];
    v = fmax(v, fmax(fabs(x.x), fabs(x.y)));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  __shared__ double wmax[4];
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    v = fmax(fmax(wmax[0], wmax[1]), fmax(wmax[2], wmax[3]));
    if (v > 0.0) atomicMax(mxb + blockIdx.y, (unsigned long long)__double_as_longlong(v));
  }
}

// the exact power of two that brings the largest entry into [0.5, 1) when it
// lies outside [2^-256, 2^256], else 1 (no change in the usual range)
__device__ __forceinline__ double qr_scale_of(unsigned long long bits) {
  const double mx = __longlong_as_double((long long)bits);
  if (!(mx > 0.0) || !isfinite(mx) || (mx >= 0x1p-256 && mx <= 0x1p256)) return 1.0;
  int e;
  frexp(mx, &e);
  return ldexp(1.0, -e);
}

// column-major copy times the matrix's scale: W[j*m + i] = scl A[i*lda + j]
__global__ void k_to_colmajor(int64_t m, int64_t n, const double2* __restrict__ a, int64_t lda,
                              double2* __restrict__ w, int64_t sa, int64_t sw,
                              const unsigned long long* __restrict__ mxb, double* __restrict__ scl) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const double sc = qr_scale_of(mxb[blockIdx.y]);
  if (t == 0) scl[blockIdx.y] = sc;
  if (t >= m * n) return;
  a += blockIdx.y * sa;
  w += blockIdx.y * sw;
  int64_t i = t / n, j = t % n;
  const double2 x = a[i * lda + j];
  w[j * m + i] = make_double2(x.x * sc, x.y * sc);
}

// The three launches above in one for a matrix of at most QR_IN_MAX entries: one workgroup
// per matrix holds it in registers between the maximum and the copy.
constexpr int64_t QR_IN_MAX = 8192;
__global__ __launch_bounds__(1024) void k_qr_in(int m, int n, const double2* __restrict__ a,
                                                int64_t lda, double2* __restrict__ w, int64_t sa,
                                                int64_t sw, double* __restrict__ scl) {
  constexpr int E = QR_IN_MAX / 1024;
  __shared__ double wmax[16];
  a += blockIdx.x * sa;
  w += blockIdx.x * sw;
  const int t = threadIdx.x, nw = blockDim.x >> 6;
  double2 x[E];
  double v = 0.0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int at = t + e * (int)blockDim.x;
    x[e] = at < m * n ? a[(int64_t)(at / n) * lda + at % n] : make_double2(0.0, 0.0);
    v = fmax(v, fmax(fabs(x[e].x), fabs(x[e].y)));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  if ((t & 63) == 0) wmax[t >> 6] = v;
  __syncthreads();
  v = 0.0;
  for (int k = 0; k < nw; ++k) v = fmax(v, wmax[k]);
  const double sc = qr_scale_of((unsigned long long)__double_as_longlong(v));
  if (t == 0) scl[blockIdx.x] = sc;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int at = t + e * (int)blockDim.x;
    if (at < m * n) w[(int64_t)(at % n) * m + at / n] = make_double2(x[e].x * sc, x[e].y * sc);
  }
}

// reflector j, applied to column c = j + blockIdx.x (< pe) of the panel.
// Workgroup 0 stores v_j (with the unit and the zeros above), tau_j and R[j, j];
// column j of W itself is left as it is (rows > j are not read again).
__global__ __launch_bounds__(256) void k_qr_col(int64_t m, int64_t j, double2* __restrict__ W,
                                                double2* __restrict__ Vf,
                                                double2* __restrict__ tau,
                                                double2* __restrict__ rdiag, QrStrides bs) {
  W += blockIdx.y * bs.W;
  Vf += blockIdx.y * bs.V;
  tau += blockIdx.y * bs.k;
  rdiag += blockIdx.y * bs.k;
  const double2* xj = W + j * m;
  const double2 alpha = xj[j];
  double s = 0;
  for (int64_t i = j + 1 + threadIdx.x; i < m; i += 256) {
    const double2 x = xj[i];
    s += x.x * x.x + x.y * x.y;
  }
  double unused = 0;
  block_sum2(s, unused);
  const double xnorm = sqrt(s);
  double2* vj = Vf + j * m;
  if (xnorm == 0.0 && alpha.y == 0.0) {
    // H_j = I: the other columns are unchanged
    if (blockIdx.x == 0) {
      for (int64_t i = threadIdx.x; i < m; i += 256)
        vj[i] = make_double2(i == j ? 1.0 : 0.0, 0.0);
      if (threadIdx.x == 0) {
        tau[j] = make_double2(0.0, 0.0);
        rdiag[j] = alpha;
      }
    }
    return;
  }
  // |(alpha_r, alpha_i, xnorm)| with scaling against overflow
  const double ar = fabs(alpha.x), ai = fabs(alpha.y);
  const double mx = fmax(fmax(ar, ai), xnorm);
  const double nrm = mx * sqrt((ar / mx) * (ar / mx) + (ai / mx) * (ai / mx) +
                               (xnorm / mx) * (xnorm / mx));
  const double beta = -copysign(nrm, alpha.x);
  // v_i = x_i / (alpha - beta) for i > j
  const double dr = alpha.x - beta, di = alpha.y;
  const double den = dr * dr + di * di;
  const double sr = dr / den, si = -di / den;
  const double2 t = make_double2((beta - alpha.x) / beta, -alpha.y / beta);
  if (blockIdx.x == 0) {
    for (int64_t i = threadIdx.x; i < m; i += 256) {
      double2 v;
      if (i < j) v = make_double2(0.0, 0.0);
      else if (i == j) v = make_double2(1.0, 0.0);
      else { const double2 x = xj[i]; v = make_double2(x.x * sr - x.y * si, x.x * si + x.y * sr); }
      vj[i] = v;
    }
    if (threadIdx.x == 0) {
      tau[j] = t;
      rdiag[j] = make_double2(beta, 0.0);
    }
    return;
  }
  // column c: w = v^H x, x <- x - conj(tau) w v (rows >= j)
  double2* xc = W + (j + blockIdx.x) * m;
  double wr = 0, wi = 0;
  for (int64_t i = j + threadIdx.x; i < m; i += 256) {
    double2 v;
    if (i == j) v = make_double2(1.0, 0.0);
    else { const double2 x = xj[i]; v = make_double2(x.x * sr - x.y * si, x.x * si + x.y * sr); }
    const double2 xi = xc[i];
    wr += v.x * xi.x + v.y * xi.y;
    wi += v.x * xi.y - v.y * xi.x;
  }
  block_sum2(wr, wi);
  const double fr = t.x * wr + t.y * wi, fi = t.x * wi - t.y * wr;   // conj(tau) w
  for (int64_t i = j + threadIdx.x; i < m; i += 256) {
    double2 v;
    if (i == j) v = make_double2(1.0, 0.0);
    else { const double2 x = xj[i]; v = make_double2(x.x * sr - x.y * si, x.x * si + x.y * sr); }
    double2 xi = xc[i];
    xi.x -= v.x * fr - v.y * fi;
    xi.y -= v.x * fi + v.y * fr;
    xc[i] = xi;
  }
}

// reflectors j and j+1 in one launch; workgroup b handles column c = j + b.
// Every workgroup forms reflector j from column j, applies it to column j+1
// on the fly (y = H_j^H x_{j+1}, never stored) and forms reflector j+1 from y,
// all with the same deterministic reductions. Workgroup 0 stores v_j, tau_j
// and R[j][j]; workgroup 1 stores v_{j+1}, tau_{j+1}, R[j+1][j+1] and R[j][j+1]
// (into rsup: columns j and j+1 of W are read by every workgroup during the
// launch and are not written); workgroups b >= 2 apply H_j^H then H_{j+1}^H to
// their column.
__global__ __launch_bounds__(256) void k_qr_col2(int64_t m, int64_t j, double2* __restrict__ W,
                                                 double2* __restrict__ Vf,
                                                 double2* __restrict__ tau,
                                                 double2* __restrict__ rdiag,
                                                 double2* __restrict__ rsup, QrStrides bs) {
  W += blockIdx.y * bs.W;
  Vf += blockIdx.y * bs.V;
  tau += blockIdx.y * bs.k;
  rdiag += blockIdx.y * bs.k;
  rsup += blockIdx.y * bs.k;
  const double2* xj = W + j * m;
  const double2* xk = W + (j + 1) * m;
  const int b = blockIdx.x;
  const int t = threadIdx.x;
  double n1[1] = {0};
  for (int64_t i = j + 1 + t; i < m; i += 256) {
    const double2 x = xj[i];
    n1[0] += x.x * x.x + x.y * x.y;
  }
  block_sum<1>(n1);
  const Refl h1 = make_refl(xj[j], sqrt(n1[0]));
  auto v1 = [&](int64_t i) -> double2 {
    return i == j ? make_double2(1.0, 0.0) : cmul2(xj[i], h1.sc);   // i >= j
  };
  if (b == 0) {
    double2* vj = Vf + j * m;
    for (int64_t i = t; i < m; i += 256) vj[i] = (i < j) ? make_double2(0.0, 0.0) : v1(i);
    if (t == 0) { tau[j] = h1.tau; rdiag[j] = h1.rd; }
    return;
  }
  double2* xc = W + (j + b) * m;
  const bool own = b >= 2;
  // w1 = v1^H x_{j+1}, wc = v1^H x_c (rows >= j)
  double d2[4] = {0, 0, 0, 0};
  for (int64_t i = j + t; i < m; i += 256) {
    const double2 v = v1(i), x = xk[i];
    d2[0] += v.x * x.x + v.y * x.y;
    d2[1] += v.x * x.y - v.y * x.x;
    if (own) {
      const double2 z = xc[i];
      d2[2] += v.x * z.x + v.y * z.y;
      d2[3] += v.x * z.y - v.y * z.x;
    }
  }
  block_sum<4>(d2);
  const double2 f1 = cmul2(conj2(h1.tau), make_double2(d2[0], d2[1]));
  const double2 fc = cmul2(conj2(h1.tau), make_double2(d2[2], d2[3]));
  auto y = [&](int64_t i) -> double2 {   // H_j^H x_{j+1}, rows >= j
    const double2 v = v1(i), g = cmul2(f1, v), x = xk[i];
    return make_double2(x.x - g.x, x.y - g.y);
  };
  auto z = [&](int64_t i) -> double2 {   // H_j^H x_c, rows >= j
    const double2 v = v1(i), g = cmul2(fc, v), x = xc[i];
    return make_double2(x.x - g.x, x.y - g.y);
  };
  // |y| below row j+1, and y^H z below row j+1
  double d3[3] = {0, 0, 0};
  for (int64_t i = j + 2 + t; i < m; i += 256) {
    const double2 yi = y(i);
    d3[0] += yi.x * yi.x + yi.y * yi.y;
    if (own) {
      const double2 zi = z(i);
      d3[1] += yi.x * zi.x + yi.y * zi.y;
      d3[2] += yi.x * zi.y - yi.y * zi.x;
    }
  }
  block_sum<3>(d3);
  const double2 alpha2 = y(j + 1);
  const Refl h2 = make_refl(alpha2, sqrt(d3[0]));
  auto v2 = [&](int64_t i) -> double2 {   // i >= j+1
    return i == j + 1 ? make_double2(1.0, 0.0) : cmul2(y(i), h2.sc);
  };
  if (b == 1) {
    double2* vk = Vf + (j + 1) * m;
    for (int64_t i = t; i < m; i += 256) vk[i] = (i <= j) ? make_double2(0.0, 0.0) : v2(i);
    if (t == 0) { tau[j + 1] = h2.tau; rdiag[j + 1] = h2.rd; rsup[j] = y(j); }
    return;
  }
  // w2 = v2^H z = z_{j+1} + conj(sc2) (y^H z)_{> j+1};  x_c <- z - conj(tau2) w2 v2
  const double2 zk = (j + 1 < m) ? z(j + 1) : make_double2(0.0, 0.0);
  const double2 yz = cmul2(conj2(h2.sc), make_double2(d3[1], d3[2]));
  const double2 f2 = cmul2(conj2(h2.tau), make_double2(zk.x + yz.x, zk.y + yz.y));
  __syncthreads();   // every thread has read row j+1 of x_c (zk) before it is overwritten
  // every row is read into registers before the row is written (same thread)
  for (int64_t i = j + t; i < m; i += 256) {
    double2 o = z(i);
    if (i >= j + 1) {
      const double2 g = cmul2(f2, v2(i));
      o.x -= g.x;
      o.y -= g.y;
    }
    xc[i] = o;
  }
}

// k_qr_col2 with the rows j .. m-1 of the three columns held in registers
// (row j + t + 256 u in thread t, u < R; requires m - j <= 256 R): one load of
// each column instead of one per pass. Every workgroup of a launch runs the
// same reductions in the same order, so the reflectors agree bitwise across
// workgroups (the grouping of rows per thread differs from k_qr_col2, so the
// two kernels agree to rounding).
template <int R>
__global__ __launch_bounds__(256) void k_qr_col2r(int64_t m, int64_t j, double2* __restrict__ W,
                                                  double2* __restrict__ Vf,
                                                  double2* __restrict__ tau,
                                                  double2* __restrict__ rdiag,
                                                  double2* __restrict__ rsup, QrStrides bs) {
  W += blockIdx.y * bs.W;
  Vf += blockIdx.y * bs.V;
  tau += blockIdx.y * bs.k;
  rdiag += blockIdx.y * bs.k;
  rsup += blockIdx.y * bs.k;
  const double2* xj = W + j * m;
  const double2* xk = W + (j + 1) * m;
  const int b = blockIdx.x;
  const int t = threadIdx.x;
  double2* xc = W + (j + b) * m;
  const bool own = b >= 2;
  double2 rj[R], rk[R], rc[R];
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int64_t i = j + t + 256 * u;
    const bool in = i < m;
    rj[u] = in ? xj[i] : make_double2(0.0, 0.0);
    rk[u] = (in && b >= 1) ? xk[i] : make_double2(0.0, 0.0);
    rc[u] = (in && own) ? xc[i] : make_double2(0.0, 0.0);
  }
  const double2 aj = xj[j];
  double n1[1] = {0};
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int64_t i = j + t + 256 * u;
    if (i > j && i < m) n1[0] += rj[u].x * rj[u].x + rj[u].y * rj[u].y;
  }
  block_sum<1>(n1);
  const Refl h1 = make_refl(aj, sqrt(n1[0]));
  auto v1r = [&](int u, int64_t i) -> double2 {
    return i == j ? make_double2(1.0, 0.0) : cmul2(rj[u], h1.sc);
  };
  if (b == 0) {
    double2* vj = Vf + j * m;
    for (int64_t i = t; i < j; i += 256) vj[i] = make_double2(0.0, 0.0);
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int64_t i = j + t + 256 * u;
      if (i < m) vj[i] = v1r(u, i);
    }
    if (t == 0) { tau[j] = h1.tau; rdiag[j] = h1.rd; }
    return;
  }
  double d2[4] = {0, 0, 0, 0};
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int64_t i = j + t + 256 * u;
    if (i < m) {
      const double2 v = v1r(u, i), x = rk[u];
      d2[0] += v.x * x.x + v.y * x.y;
      d2[1] += v.x * x.y - v.y * x.x;
      if (own) {
        const double2 z = rc[u];
        d2[2] += v.x * z.x + v.y * z.y;
        d2[3] += v.x * z.y - v.y * z.x;
      }
    }
  }
  block_sum<4>(d2);
  const double2 f1 = cmul2(conj2(h1.tau), make_double2(d2[0], d2[1]));
  const double2 fc = cmul2(conj2(h1.tau), make_double2(d2[2], d2[3]));
  double2 y[R], z[R];
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int64_t i = j + t + 256 * u;
    const double2 v = v1r(u, i), g = cmul2(f1, v), gc = cmul2(fc, v);
    y[u] = make_double2(rk[u].x - g.x, rk[u].y - g.y);
    z[u] = make_double2(rc[u].x - gc.x, rc[u].y - gc.y);
  }
  double d3[3] = {0, 0, 0};
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int64_t i = j + t + 256 * u;
    if (i >= j + 2 && i < m) {
      d3[0] += y[u].x * y[u].x + y[u].y * y[u].y;
      if (own) {
        d3[1] += y[u].x * z[u].x + y[u].y * z[u].y;
        d3[2] += y[u].x * z[u].y - y[u].y * z[u].x;
      }
    }
  }
  block_sum<3>(d3);
  // rows j and j+1 of y and z from memory (every thread needs them)
  auto yg = [&](int64_t i) -> double2 {
    const double2 v = i == j ? make_double2(1.0, 0.0) : cmul2(xj[i], h1.sc), g = cmul2(f1, v),
                  x = xk[i];
    return make_double2(x.x - g.x, x.y - g.y);
  };
  const double2 alpha2 = yg(j + 1);
  const Refl h2 = make_refl(alpha2, sqrt(d3[0]));
  if (b == 1) {
    double2* vk = Vf + (j + 1) * m;
    for (int64_t i = t; i <= j; i += 256) vk[i] = make_double2(0.0, 0.0);
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int64_t i = j + t + 256 * u;
      if (i > j && i < m) vk[i] = i == j + 1 ? make_double2(1.0, 0.0) : cmul2(y[u], h2.sc);
    }
    if (t == 0) { tau[j + 1] = h2.tau; rdiag[j + 1] = h2.rd; rsup[j] = yg(j); }
    return;
  }
  // w2 = v2^H z = z_{j+1} + conj(sc2) (y^H z)_{> j+1};  x_c <- z - conj(tau2) w2 v2
  double2 zk = make_double2(0.0, 0.0);
  if (j + 1 < m) {
    const double2 v = cmul2(xj[j + 1], h1.sc), g = cmul2(fc, v), x = xc[j + 1];
    zk = make_double2(x.x - g.x, x.y - g.y);
  }
  const double2 yz = cmul2(conj2(h2.sc), make_double2(d3[1], d3[2]));
  const double2 f2 = cmul2(conj2(h2.tau), make_double2(zk.x + yz.x, zk.y + yz.y));
  __syncthreads();   // every thread has read row j+1 of x_c (zk) before it is overwritten
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int64_t i = j + t + 256 * u;
    if (i < m) {
      double2 o = z[u];
      if (i >= j + 1) {
        const double2 v2 = i == j + 1 ? make_double2(1.0, 0.0) : cmul2(y[u], h2.sc);
        const double2 g = cmul2(f2, v2);
        o.x -= g.x;
        o.y -= g.y;
      }
      xc[i] = o;
    }
  }
}

// G[a][b] = v_a^H v_b (a <= b in steps of 16) of the panel's reflectors over the rows
// first .. end - 1: FP64 MFMA on 16 x 16 tiles, the operands loaded as in the
// cross Gram kernel of the Jacobi iteration (a lane holds rows 2 kk, 2 kk + 1 of every 8
// of column l16); columns >= nbp count as zero. Thread t (of 256) ends with entry (t / 16,
// t % 16) of the tiles (0, 0), (0, 16) and (16, 16). No __restrict__ here: k_qr_panel reads
// what its own waves have just stored.
typedef double2 VtvRed[4][3][4][64];
__device__ __forceinline__ void vtv_block(int64_t m, int64_t j0, int nbp, int64_t first,
                                          int64_t end, const double2* Vf,
                                          VtvRed& red, double2 (&g)[3]) {
  static_assert(QR_NB == 32, "two 16-column tiles");
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int l16 = lane & 15, kk = lane >> 4;
  d4_t re[3], im[3];
#pragma unroll
  for (int h = 0; h < 3; ++h) re[h] = im[h] = d4_t{0, 0, 0, 0};
  const double2* V0 = Vf + (j0 + l16) * m;
  const double2* V1 = V0 + 16 * m;
  const bool in0 = l16 < nbp, in1 = 16 + l16 < nbp;
  for (int64_t r0 = first + 32 * wave; r0 < end; r0 += 128) {
    double2 a[4][2], b[4][2];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int64_t i = r0 + 8 * u + 2 * kk + h;
        a[u][h] = (in0 && i < end) ? V0[i] : make_double2(0.0, 0.0);
        b[u][h] = (in1 && i < end) ? V1[i] : make_double2(0.0, 0.0);
      }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const double2 x[3] = {a[u][h], a[u][h], b[u][h]}, y[3] = {a[u][h], b[u][h], b[u][h]};
#pragma unroll
        for (int e = 0; e < 3; ++e) {
          re[e] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[e].x, y[e].x, re[e], 0, 0, 0);
          im[e] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[e].x, y[e].y, im[e], 0, 0, 0);
          re[e] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[e].y, y[e].y, re[e], 0, 0, 0);
          im[e] = __builtin_amdgcn_mfma_f64_16x16x4f64(-x[e].y, y[e].x, im[e], 0, 0, 0);
        }
      }
  }
#pragma unroll
  for (int e = 0; e < 3; ++e)
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave][e][v][lane] = make_double2(re[e][v], im[e][v]);
  __syncthreads();
  const int i = t >> 4, j = t & 15, src = 16 * (i & 3) + j;
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    g[e] = make_double2(0.0, 0.0);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const double2 v = red[w][e][i >> 2][src];
      g[e].x += v.x;
      g[e].y += v.y;
    }
  }
}

// compact WY factor (forward, columnwise; zero padded to QR_NB x QR_NB): T of a
// single reflector is tau, and two neighbouring blocks combine to
//   T = [[T1, -T1 (V1^H V2) T2], [0, T2]],
// so five levels of doubling build the factor with all threads at work (a column by
// column recurrence in one wave took 19 us). Gs holds V^H V above the diagonal and zeros
// elsewhere.
typedef double2 QrTile[QR_NB][QR_NB + 1];
__device__ __forceinline__ void tmat_block(int nbp, const QrTile& Gs, QrTile& Ts, QrTile& Ms,
                                           const double2* tau, double2* T) {
  const int t = threadIdx.x;
#pragma unroll
  for (int u = 0; u < QR_NB * QR_NB / 256; ++u) {
    const int e = t + 256 * u, a = e / QR_NB, b = e % QR_NB;
    Ts[a][b] = (a == b && a < nbp) ? tau[a] : make_double2(0.0, 0.0);
  }
  __syncthreads();
#pragma unroll
  for (int h = 1; h < QR_NB; h *= 2) {
    // output (i, j) of block pair b: 16 h outputs in all
    const int b = t / (h * h), i = (t / h) % h, j = t % h;
    const int r0 = 2 * h * b, c0 = r0 + h;
    const bool on = t < 16 * h;
    if (on) {   // M = (V1^H V2) T2
      double2 m = make_double2(0.0, 0.0);
#pragma unroll
      for (int k = 0; k < h; ++k) {
        const double2 x = cmul2(Gs[r0 + i][c0 + k], Ts[c0 + k][c0 + j]);
        m.x += x.x;
        m.y += x.y;
      }
      Ms[r0 + i][c0 + j] = m;
    }
    __syncthreads();
    if (on) {
      double2 m = make_double2(0.0, 0.0);
#pragma unroll
      for (int k = 0; k < h; ++k) {
        const double2 x = cmul2(Ts[r0 + i][r0 + k], Ms[r0 + k][c0 + j]);
        m.x -= x.x;
        m.y -= x.y;
      }
      Ts[r0 + i][c0 + j] = m;
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < QR_NB * QR_NB / 256; ++u) {
    const int e = t + 256 * u;
    T[e] = Ts[e / QR_NB][e % QR_NB];
  }
}

// V^H V over the rows j0 + rows blockIdx.x .. (rows a multiple of 128) as a partial G, and
// T from the sum of the partials (eight of them 11.1 us one load after the other, 6.2 at once): panels of more than 256 rows (shorter ones: k_qr_panel)
__global__ __launch_bounds__(256) void k_qr_vtv(int64_t m, int64_t j0, int nbp, int rows,
                                                const double2* __restrict__ Vf,
                                                double2* __restrict__ G, QrStrides bs) {
  __shared__ VtvRed red;
  Vf += blockIdx.y * bs.V;
  G += blockIdx.y * bs.G + (int64_t)blockIdx.x * QR_NB * QR_NB;
  const int64_t first = j0 + (int64_t)blockIdx.x * rows;
  double2 g[3];
  vtv_block(m, j0, nbp, first, first + rows < m ? first + rows : m, Vf, red, g);
  const int i = threadIdx.x >> 4, j = threadIdx.x & 15;
#pragma unroll
  for (int e = 0; e < 3; ++e)
    G[((e == 2 ? 16 : 0) + i) * QR_NB + (e == 0 ? 0 : 16) + j] = g[e];
}
__global__ __launch_bounds__(256) void k_qr_tmat(int nbp, int nparts, const double2* __restrict__ G,
                                                 const double2* __restrict__ tau,
                                                 double2* __restrict__ T, QrStrides bs) {
  __shared__ QrTile Gs, Ts, Ms;
  G += blockIdx.x * bs.G + threadIdx.x;
  constexpr int E = QR_NB * QR_NB / 256;
  double2 g[E];
#pragma unroll
  for (int u = 0; u < E; ++u) g[u] = make_double2(0.0, 0.0);
#pragma unroll 8
  for (int p = 0; p < nparts; ++p)   // all loads in flight at once
#pragma unroll
    for (int u = 0; u < E; ++u) {
      const double2 v = G[(int64_t)p * QR_NB * QR_NB + 256 * u];
      g[u].x += v.x;
      g[u].y += v.y;
    }
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int e = threadIdx.x + 256 * u, a = e / QR_NB, b = e % QR_NB;
    // (below the diagonal blocks and beyond nbp G is not written or not used)
    Gs[a][b] = a < b && b < nbp ? g[u] : make_double2(0.0, 0.0);
  }
  tmat_block(nbp, Gs, Ts, Ms, tau + blockIdx.x * bs.k, T + blockIdx.x * bs.T);
}

// A whole panel of at most 64 R rows factored by one workgroup with its columns
// j0 .. j0+nbp-1 (nbp <= C NW) in registers: column j0 + q NW + w in element q of
// wave w, row j0 + lane + 64 u in element u. The current column y is read from
// LDS (two buffers, one barrier per column) as it stands before its reflector is
// known: every wave forms |y|^2 and the products y^H x with its own columns in the
// same pass, sums them inside the wave and derives the reflector itself,
//   v = [1, sc y],  x_j -= f,  x -= f sc y  with  f = conj(tau) (x_j + conj(sc) y^H x),
// so the chain per column is one pass, one sum and one update. Bound by the
// instructions of one CU: 32 columns of 256 rows take 60 us with T (48 before, 95 with two
// columns per launch), of 128 rows 48, of 64 rows 43; up to 16 columns of 64 rows 16 us with four
// columns per wave (22 with eight, half of them empty).
// Writes v_j (rows >= j0), tau_j, R[j][j], the rows j0 .. j-1 of R above it, and the panel's
// T (about 12 us, as long as the two launches that form it for longer panels, without the gaps).
template <int R, int C, int NW>
__global__ __launch_bounds__(64 * NW) void k_qr_panel(int64_t m, int64_t j0, int nbp,
                                                      double2* __restrict__ W,
                                                      double2* __restrict__ Vf,
                                                      double2* __restrict__ tau,
                                                      double2* __restrict__ rdiag,
                                                      double2* __restrict__ T, QrStrides bs) {
  static_assert(NW == 4, "256 threads");
  struct TPart {
    QrTile Ts, Ms;
  };
  __shared__ __align__(16) union {
    double2 Ys[2][64 * R];
    VtvRed red;
    TPart tp;
  } sm;
  __shared__ QrTile Gs;
  auto& Ys = sm.Ys;
  W += blockIdx.x * bs.W;
  Vf += blockIdx.x * bs.V;
  tau += blockIdx.x * bs.k;
  rdiag += blockIdx.x * bs.k;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double2 x[C][R];
#pragma unroll
  for (int q = 0; q < C; ++q) {
    const int c = q * NW + wave;
    const double2* src = W + (j0 + c) * m;
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int64_t i = j0 + lane + 64 * u;
      x[q][u] = (c < nbp && i < m) ? src[i] : make_double2(0.0, 0.0);
    }
  }
  if (wave == 0) {
#pragma unroll
    for (int u = 0; u < R; ++u) Ys[0][64 * u + lane] = x[0][u];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < C; ++q) {
    for (int wo = 0; wo < NW; ++wo) {
      const int jj = q * NW + wo;
      if (jj >= nbp) break;
      const int buf = jj & 1;
      const double2 alpha = Ys[buf][jj];
      double2 y[R];
#pragma unroll
      for (int u = 0; u < R; ++u) y[u] = Ys[buf][64 * u + lane];
      if (lane <= jj) y[0] = make_double2(0.0, 0.0);
      double s2 = 0.0, dr[C] = {}, di[C] = {};
#pragma unroll
      for (int u = 0; u < R; ++u) s2 += y[u].x * y[u].x + y[u].y * y[u].y;
#pragma unroll
      for (int p = q; p < C; ++p) {
        dr[p] = di[p] = 0.0;
#pragma unroll
        for (int u = 0; u < R; ++u) {
          dr[p] += y[u].x * x[p][u].x + y[u].y * x[p][u].y;
          di[p] += y[u].x * x[p][u].y - y[u].y * x[p][u].x;
        }
      }
      {
        // eight sums at a time; |y|^2 takes a free slot when the first column is done
        static_assert(C % 4 == 0, "four products per group of eight sums");
        if (q == 0) s2 = wave_sum(s2);
#pragma unroll
        for (int p0 = q / 4 * 4; p0 < C; p0 += 4) {
          double v8[8];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            v8[2 * k] = p0 + k >= q ? dr[p0 + k] : (p0 + k == q - 1 ? s2 : 0.0);
            v8[2 * k + 1] = p0 + k >= q ? di[p0 + k] : 0.0;
          }
          const double sums = wave_sum8(v8);
          if (q > 0 && q % 4 != 0 && p0 < q) s2 = lane_value(sums, 8 * sum8_slot(2 * (q - 1 - p0)));
          if (q > 0 && q % 4 == 0 && p0 == q) s2 = wave_sum(s2);
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (p0 + k >= q) {
              dr[p0 + k] = lane_value(sums, 8 * sum8_slot(2 * k));
              di[p0 + k] = lane_value(sums, 8 * sum8_slot(2 * k + 1));
            }
        }
      }
      const Refl h = make_refl2(alpha, s2);
      // later columns (element q only of the waves after the owner)
#pragma unroll
      for (int p = q; p < C; ++p) {
        const double2 xj = make_double2(lane_value(x[p][0].x, jj), lane_value(x[p][0].y, jj));
        const double2 d = cmul2(conj2(h.sc), make_double2(dr[p], di[p]));
        double2 f = cmul2(conj2(h.tau), make_double2(xj.x + d.x, xj.y + d.y));
        if (p == q && wave <= wo) f = make_double2(0.0, 0.0);
        const double2 g = cmul2(f, h.sc);
#pragma unroll
        for (int u = 0; u < R; ++u) {
          x[p][u].x -= g.x * y[u].x - g.y * y[u].y;
          x[p][u].y -= g.x * y[u].y + g.y * y[u].x;
        }
        if (lane == jj) {
          x[p][0].x -= f.x;
          x[p][0].y -= f.y;
        }
        // the next column goes out first
        if (p == q + (wo == NW - 1) && wave == (wo + 1) % NW) {
#pragma unroll
          for (int u = 0; u < R; ++u) Ys[buf ^ 1][64 * u + lane] = x[p][u];
        }
      }
      if (wave == wo) {
        double2* vj = Vf + (j0 + jj) * m;
#pragma unroll
        for (int u = 0; u < R; ++u) {
          const int64_t i = j0 + lane + 64 * u;
          double2 v = cmul2(y[u], h.sc);
          if (u == 0 && lane == jj) v = make_double2(1.0, 0.0);
          if (i < m) vj[i] = v;
        }
        if (lane < jj) W[(j0 + jj) * m + j0 + lane] = x[q][0];   // finished rows of R
        if (lane == 0) {
          tau[j0 + jj] = h.tau;
          rdiag[j0 + jj] = h.rd;
        }
      }
      __syncthreads();
    }
  }
  // V^H V and T (the barrier above orders the stores of V and tau with these loads)
  double2 g[3];
  vtv_block(m, j0, nbp, j0, m, Vf, sm.red, g);
  const int gi = threadIdx.x >> 4, gj = threadIdx.x & 15;
  const double2 zero = make_double2(0.0, 0.0);
  Gs[gi][gj] = gi < gj && gj < nbp ? g[0] : zero;
  Gs[gi][16 + gj] = 16 + gj < nbp ? g[1] : zero;
  Gs[16 + gi][gj] = zero;
  Gs[16 + gi][16 + gj] = gi < gj && 16 + gj < nbp ? g[2] : zero;
  __syncthreads();
  tmat_block(nbp, Gs, sm.tp.Ts, sm.tp.Ms, tau + j0, T + blockIdx.x * bs.T);
}

// Columns j .. j+nc-1 (nc <= 4) of a panel that starts at j0, at most 256 R rows below j,
// in one launch: workgroup b handles column j + b. Every workgroup factors the nc
// columns for itself in registers (row j + t + 256 u in element u of thread t; the
// same reductions in the same order, so the reflectors agree bitwise), each with
// one reduction over the workgroup: |y|^2 and the products y^H x with the columns that
// follow, before the reflector is known (as in k_qr_panel). Workgroups b < nc
// store v_{j+b}, tau, R[j+b][j+b] and, into rup (QR_NB x QR_NB, panel-local), the
// rows j .. j+b-1 of R above it: the columns j .. j+nc-1 of W are read by every
// workgroup during the launch and are not written. The others apply the
// reflectors to their column. 8 rows per thread (2048 rows): 7.9 us for four columns, against
// 14.8 for two launches of two columns; 4 rows: 6.5 against 12.8; 2 rows: 5.6.
template <int R>
__global__ __launch_bounds__(256) void k_qr_col4(int64_t m, int64_t j0, int64_t j, int nc,
                                                 double2* __restrict__ W,
                                                 double2* __restrict__ Vf,
                                                 double2* __restrict__ tau,
                                                 double2* __restrict__ rdiag,
                                                 double2* __restrict__ rup, QrStrides bs) {
  constexpr int K = 4;
  __shared__ double red[2][2 * K + 1][4];   // |y|^2, then re / im of y^H x per later column
  __shared__ double2 top[2][K + 1];         // row j + c of the columns, the own one last
  W += blockIdx.y * bs.W;
  Vf += blockIdx.y * bs.V;
  tau += blockIdx.y * bs.k;
  rdiag += blockIdx.y * bs.k;
  rup += blockIdx.y * bs.G;
  const int t = threadIdx.x, wave = t >> 6, b = blockIdx.x;
  const bool own = b >= nc;
  double2 x[K + 1][R];
#pragma unroll
  for (int c = 0; c <= K; ++c) {
    const int64_t col = c < K ? j + c : j + b;
    const bool on = c < K ? c < nc : own;
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int64_t i = j + t + 256 * u;
      x[c][u] = (on && i < m) ? W[col * m + i] : make_double2(0.0, 0.0);
    }
  }
  Refl mine = {};
#pragma unroll
  for (int c = 0; c < K; ++c) {
    if (c < nc) {
      const double2 y0 = t > c ? x[c][0] : make_double2(0.0, 0.0);
      double s[2 * K + 1];
#pragma unroll
      for (int v = 0; v < 2 * K + 1; ++v) s[v] = 0.0;
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const double2 y = u == 0 ? y0 : x[c][u];
        s[0] += y.x * y.x + y.y * y.y;
#pragma unroll
        for (int p = c + 1; p <= K; ++p) {
          s[2 * p - 1] += y.x * x[p][u].x + y.y * x[p][u].y;
          s[2 * p] += y.x * x[p][u].y - y.y * x[p][u].x;
        }
      }
      {
        // eight products (the slots of finished columns are free: |y|^2 takes one)
        double v8[8];
#pragma unroll
        for (int v = 0; v < 8; ++v) v8[v] = v + 1 > 2 * c ? s[v + 1] : (v == 0 ? s[0] : 0.0);
        const double sums = wave_sum8(v8);
        const int slot = sum8_slot((t & 63) >> 3);
        if ((t & 7) == 0) red[c & 1][c > 0 && slot == 0 ? 0 : slot + 1][wave] = sums;
        if (c == 0) {
          const double r = wave_sum(s[0]);
          if ((t & 63) == 0) red[0][0][wave] = r;
        }
      }
      if (t == c) {
#pragma unroll
        for (int p = c; p <= K; ++p) top[c & 1][p] = x[p][0];
      }
      __syncthreads();
#pragma unroll
      for (int v = 0; v < 2 * K + 1; ++v)
        if (v == 0 || v > 2 * c) {
          const double* r = red[c & 1][v];
          s[v] = (r[0] + r[1]) + (r[2] + r[3]);
        }
      const Refl h = make_refl2(top[c & 1][c], s[0]);
      if (b == c) mine = h;
#pragma unroll
      for (int p = c + 1; p <= K; ++p) {
        const double2 xj = top[c & 1][p];
        const double2 d = cmul2(conj2(h.sc), make_double2(s[2 * p - 1], s[2 * p]));
        const double2 f = cmul2(conj2(h.tau), make_double2(xj.x + d.x, xj.y + d.y));
        const double2 g = cmul2(f, h.sc);
#pragma unroll
        for (int u = 0; u < R; ++u) {
          const double2 y = u == 0 ? y0 : x[c][u];
          x[p][u].x -= g.x * y.x - g.y * y.y;
          x[p][u].y -= g.x * y.y + g.y * y.x;
        }
        if (t == c) {
          x[p][0].x -= f.x;
          x[p][0].y -= f.y;
        }
      }
    }
  }
  if (own) {
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int64_t i = j + t + 256 * u;
      if (i < m) W[(j + b) * m + i] = x[K][u];
    }
    return;
  }
  double2* vj = Vf + (j + b) * m;
  for (int64_t i = j0 + t; i < j; i += 256) vj[i] = make_double2(0.0, 0.0);
#pragma unroll
  for (int c = 0; c < K; ++c) {
    if (c == b) {
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const int64_t i = j + t + 256 * u;
        double2 v = cmul2(x[c][u], mine.sc);
        if (u == 0 && t <= c) v = make_double2(t == c ? 1.0 : 0.0, 0.0);
        if (i < m) vj[i] = v;
      }
      if (t < c) rup[(j - j0 + t) * QR_NB + (j - j0 + c)] = x[c][0];
      if (t == 0) {
        tau[j + c] = mine.tau;
        rdiag[j + c] = mine.rd;
      }
    }
  }
}

// the entries of R inside the groups of four columns of a panel, from rup into W
// after the panel
__global__ void k_qr_fixup4(int64_t m, int64_t j0, int nbp, const double2* __restrict__ rup,
                            double2* __restrict__ W, QrStrides bs) {
  rup += blockIdx.x * bs.G;
  W += blockIdx.x * bs.W;
  for (int e = threadIdx.x; e < QR_NB * QR_NB; e += 256) {
    const int a = e / QR_NB, b = e % QR_NB;
    if (a < b && b < nbp && a / 4 == b / 4) W[(j0 + b) * m + j0 + a] = rup[e];
  }
}

// R[jj][jj+1] of the two-reflector launches of a panel, written after the panel
__global__ void k_qr_fixsup(int64_t m, int64_t j0, int64_t pe, const double2* __restrict__ rsup,
                            double2* __restrict__ W, QrStrides bs) {
  rsup += blockIdx.y * bs.k;
  W += blockIdx.y * bs.W;
  const int64_t jj = j0 + 2 * (int64_t)threadIdx.x;
  if (jj + 1 < pe) W[(jj + 1) * m + jj] = rsup[jj];
}

// Y = sum of the nparts partial products P[s] (QR_NB x nc, rows < nbp used);
// Z = -T^H Y (adjoint = 1) or Z = -T Y (adjoint = 0). A workgroup handles 8
// columns; thread (r, cl) sums row r of column cl, then forms row r of Z.
// (7.2 us at 1024 rows with one load and one term at a time, 4.6 with several in flight
// at once.)
static_assert(QR_NB * 8 == 256, "k_qr_reduce maps its 256 threads onto QR_NB rows x 8 columns");
__global__ __launch_bounds__(256) void k_qr_reduce(int nbp, int64_t nc, int nparts,
                                                   const double2* __restrict__ P,
                                                   const double2* __restrict__ T, int adjoint,
                                                   double2* __restrict__ Z, QrStrides bs) {
  P += blockIdx.y * bs.P;
  T += blockIdx.y * bs.T;
  Z += blockIdx.y * bs.Z;
  __shared__ double2 Ts[QR_NB][QR_NB + 1];
  __shared__ double2 Ys[8][QR_NB + 1];
  const int t = threadIdx.x;
  for (int e = t; e < QR_NB * QR_NB; e += 256) Ts[e / QR_NB][e % QR_NB] = T[e];
  const int cl = t & 7, r = t >> 3;
  const int64_t c = (int64_t)blockIdx.x * 8 + cl;
  const bool ok = c < nc && r < nbp;
  double sr = 0, si = 0;
  if (ok)
#pragma unroll 8
    for (int s = 0; s < nparts; ++s) {
      const double2 v = P[((int64_t)s * QR_NB + r) * nc + c];
      sr += v.x;
      si += v.y;
    }
  Ys[cl][r] = make_double2(sr, si);
  __syncthreads();
  if (!ok) return;
  double zr = 0, zi = 0;
  // T is zero below its diagonal and, as y, beyond nbp: all 32 terms, read ahead
  if (adjoint) {
#pragma unroll 8
    for (int q = 0; q < QR_NB; ++q) {   // (T^H y)_r
      const double2 a = Ts[q][r], y = Ys[cl][q];
      zr += a.x * y.x + a.y * y.y;
      zi += a.x * y.y - a.y * y.x;
    }
  } else {
#pragma unroll 8
    for (int q = 0; q < QR_NB; ++q) {   // (T y)_r
      const double2 a = Ts[r][q], y = Ys[cl][q];
      zr += a.x * y.x - a.y * y.y;
      zi += a.x * y.y + a.y * y.x;
    }
  }
  Z[(int64_t)r * nc + c] = make_double2(-zr, -zi);
}

static inline size_t al(size_t b) { return (b + 255) & ~(size_t)255; }

// row segments of the V^H V products over `rows` rows: at least 128 rows each
static int64_t vtv_parts(int64_t rows) {
  const int64_t p = (rows + 127) / 128;
  return p < QR_VTV_PARTS ? p : QR_VTV_PARTS;
}

static QrStrides qr_strides(int64_t m, int64_t n, int64_t ncmax) {
  const int64_t k = m < n ? m : n;
  const int64_t npan = (k + QR_NB - 1) / QR_NB;
  const int64_t nc = ncmax > n ? ncmax : n;
  QrStrides b;
  b.W = m * n;
  b.V = m * k;
  b.k = k + 1;
  b.T = (npan + 1) * QR_NB * QR_NB;
  b.G = vtv_parts(m) * QR_NB * QR_NB;
  b.P = (QR_SPLITK + 1) * QR_NB * nc;
  b.Z = QR_NB * nc;
  return b;
}

size_t qr_fact_bytes(int64_t m, int64_t n, int64_t ncmax, int64_t batch) {
  const QrStrides b = qr_strides(m, n, ncmax);
  const size_t B = (size_t)batch;
  return al(B * b.W * 16) + al(B * b.V * 16) + 3 * al(B * b.k * 16) + al(B * b.T * 16) +
         al(B * b.G * 16) + al(B * b.P * 16) + al(B * b.Z * 16) + 2 * al(B * 8);
}

QrFact qr_fact_layout(int64_t m, int64_t n, int64_t ncmax, void* ws, int64_t batch) {
  QrFact f;
  f.m = m; f.n = n; f.k = m < n ? m : n;
  f.npan = (f.k + QR_NB - 1) / QR_NB;
  f.ncmax = ncmax > n ? ncmax : n;
  f.batch = batch;
  f.bs = qr_strides(m, n, ncmax);
  const size_t B = (size_t)batch;
  char* p = (char*)ws;
  f.W = (double2*)p; p += al(B * f.bs.W * 16);
  f.Vf = (double2*)p; p += al(B * f.bs.V * 16);
  f.tau = (double2*)p; p += al(B * f.bs.k * 16);
  f.rdiag = (double2*)p; p += al(B * f.bs.k * 16);
  f.rsup = (double2*)p; p += al(B * f.bs.k * 16);
  f.T = (double2*)p; p += al(B * f.bs.T * 16);
  f.G = (double2*)p; p += al(B * f.bs.G * 16);
  f.P = (double2*)p; p += al(B * f.bs.P * 16);
  f.Z = (double2*)p; p += al(B * f.bs.Z * 16);
  f.scl = (double*)p; p += al(B * 8);
  f.mxb = (unsigned long long*)p;
  return f;
}

// C <- (I - V op(T) V^H) C, op(T) = T^H (ADJ) or T, on 8 columns of C (mr rows) per workgroup:
// the product V^H C, its reduction with T and the update in one launch, for panels whose rows
// one workgroup covers in a few steps. Y = V^H C: wave w takes rows 16 (w % 2) .. of Y and
// every fourth part of the rows of C; the update goes over tiles of 16 rows. FP64 MFMA with
// the real embedding of the products (gemm_impl.h), operands straight from memory.
// Up to 256 rows (512 in a batch, whose three products fill the chip no better): QR of
// 64 x 32 67 -> 60 us, 128 x 64 152 -> 136, 256 x 128 359 -> 340, 8 of 512 x 256 1020 -> 911; one
// of 512 x 256 807 -> 815, of 1024 x 512 1927 -> 2232 without the limit.
constexpr int64_t QR_APPLY_ROWS = 256;
constexpr int QA_T = 512, QA_PARTS = QA_T / 128;
template <bool ADJ>
__global__ __launch_bounds__(QA_T) void k_qr_apply(int64_t ldv, int mr, int nbp,
                                                   const double2* __restrict__ V,
                                                   const double2* __restrict__ T,
                                                   double2* __restrict__ C, int64_t ldc, int nc,
                                                   QrStrides bs, int64_t sc) {
  constexpr int U = 4;
  __shared__ QrTile Ts;
  __shared__ __align__(16) double2 Yp[QA_PARTS][QR_NB][8], Ys[QR_NB][9], Zs[QR_NB][8];
  V += blockIdx.y * bs.V;
  T += blockIdx.y * bs.T;
  C += blockIdx.y * sc + (int64_t)blockIdx.x * 8 * ldc;
  nc -= 8 * (int)blockIdx.x;
  const int t = threadIdx.x, lane = t & 63, l16 = lane & 15, kk = lane >> 4, pb = lane & 1;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int col = min(l16 >> 1, nc - 1);
  for (int e = t; e < QR_NB * QR_NB; e += QA_T) Ts[e / QR_NB][e % QR_NB] = T[e];
  {
    const int vc = 16 * (wave & 1) + l16, part = wave >> 1;
    const bool on = vc < nbp;
    const double2* pv = V + (int64_t)(on ? vc : 0) * ldv;
    const double2* pc = C + (int64_t)col * ldc;
    const int steps = (mr + 3) / 4, per = (steps + QA_PARTS - 1) / QA_PARTS;
    const int s1 = min((part + 1) * per, steps);
    d4_t acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
    for (int s = part * per; s < s1; s += U) {
      double2 a[U], b[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int r = 4 * (s + u) + kk;
        const bool in = s + u < s1 && r < mr;
        a[u] = in && on ? pv[r] : make_double2(0.0, 0.0);
        b[u] = in ? pc[r] : make_double2(0.0, 0.0);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {   // conj(a) b
        const double br = pb ? b[u].y : b[u].x, bi = pb ? -b[u].x : b[u].y;
        acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u].x, br, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u].y, bi, acc1, 0, 0, 0);
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      double* y = (double*)&Yp[part][16 * (wave & 1) + kk + 4 * v][l16 >> 1];
      y[pb] = acc0[v] + acc1[v];
    }
  }
  __syncthreads();
  const int r = t >> 3, c = t & 7;
  if (r < QR_NB) {
    double2 y = make_double2(0.0, 0.0);
#pragma unroll
    for (int p = 0; p < QA_PARTS; ++p) {
      y.x += Yp[p][r][c].x;
      y.y += Yp[p][r][c].y;
    }
    Ys[r][c] = y;
  }
  __syncthreads();
  if (r < QR_NB) {   // Z = -op(T) Y (T is zero below the diagonal and beyond nbp)
    double zr = 0.0, zi = 0.0;
#pragma unroll 8
    for (int q = 0; q < QR_NB; ++q) {
      const double2 a = ADJ ? conj2(Ts[q][r]) : Ts[r][q], y = Ys[q][c];
      zr = fma(-a.x, y.x, fma(a.y, y.y, zr));
      zi = fma(-a.x, y.y, fma(-a.y, y.x, zi));
    }
    Zs[r][c] = make_double2(zr, zi);
  }
  __syncthreads();
  double2 z[QR_NB / 4];
#pragma unroll
  for (int u = 0; u < QR_NB / 4; ++u) z[u] = Zs[4 * u + kk][l16 >> 1];
  for (int m0 = 16 * wave; m0 < mr; m0 += 16 * (QA_T / 64)) {
    const double2* pv = V + min(m0 + l16, mr - 1);
    d4_t acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
    double2 a[QR_NB / 4];
#pragma unroll
    for (int u = 0; u < QR_NB / 4; ++u)
      a[u] = 4 * u + kk < nbp ? pv[(int64_t)(4 * u + kk) * ldv] : make_double2(0.0, 0.0);
#pragma unroll
    for (int u = 0; u < QR_NB / 4; ++u) {
      acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u].x, pb ? z[u].y : z[u].x, acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u].y, pb ? z[u].x : -z[u].y, acc1, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = m0 + kk + 4 * v;
      if (row < mr && (l16 >> 1) < nc) {
        double* o = (double*)(C + (int64_t)col * ldc + row) + pb;
        *o += acc0[v] + acc1[v];
      }
    }
  }
}

// C[j0:m, c0:c0+nc] += V_panel Z with Z = -T^(H) V_panel^H C[j0:m, c0:c0+nc]
// (C column-major with leading dimension ldc; panel columns j0 .. j0+nbp-1;
// matrix b of a batch at C + b * sc). A single matrix splits the K = m - j0
// rows of V^H C into chunks (batched product) for parallelism; a batch of
// matrices is batched over the matrices instead.
static int apply_block(const QrFact& f, int64_t j0, int nbp, const double2* Tp, int adjoint,
                       double2* C, int64_t ldc, int64_t c0, int64_t nc, hipStream_t s,
                       int64_t sc) {
  const int64_t m = f.m, mr = m - j0;
  if (nc <= 0 || mr <= 0) return PTN_OK;
  const double2* V = f.Vf + j0 * m + j0;
  double2* Cs = C + c0 * ldc + j0;
  if (mr <= (f.batch > 1 ? 2 * QR_APPLY_ROWS : QR_APPLY_ROWS)) {
    const dim3 g((unsigned)((nc + 7) / 8), (unsigned)f.batch);
    if (adjoint)
      k_qr_apply<true><<<g, QA_T, 0, s>>>(m, (int)mr, nbp, V, Tp, Cs, ldc, (int)nc, f.bs, sc);
    else
      k_qr_apply<false><<<g, QA_T, 0, s>>>(m, (int)mr, nbp, V, Tp, Cs, ldc, (int)nc, f.bs, sc);
    PTN_LAUNCH_CHECK();
    return PTN_OK;
  }
  int st;
  int nparts;
  if (f.batch == 1) {
    // partials P[s] = V^H C over K chunks of `chunk` rows
    int64_t chunk = (mr + QR_SPLITK - 1) / QR_SPLITK;
    chunk = ((chunk + 7) / 8) * 8;
    const int64_t nfull = mr / chunk, rem = mr - nfull * chunk;
    if (nfull > 0) {
      ZGemm g = {nbp, nc, chunk, V, m, 1, 1, Cs, 1, ldc, 0, f.P, nc, 1, 0,
                 nfull, chunk, chunk, (int64_t)QR_NB * nc};
      if ((st = zgemm(g, PTN_FP64, PTN_T_C128, PTN_T_C128, PTN_T_C128, nullptr, 0, s))) return st;
    }
    if (rem > 0) {
      ZGemm g = {nbp, nc, rem, V + nfull * chunk, m, 1, 1, Cs + nfull * chunk, 1, ldc, 0,
                 f.P + nfull * QR_NB * nc, nc, 1, 0, 1, 0, 0, 0};
      if ((st = zgemm(g, PTN_FP64, PTN_T_C128, PTN_T_C128, PTN_T_C128, nullptr, 0, s))) return st;
    }
    nparts = (int)(nfull + (rem > 0 ? 1 : 0));
  } else {
    ZGemm g = {nbp, nc, mr, V, m, 1, 1, Cs, 1, ldc, 0, f.P, nc, 1, 0,
               f.batch, f.bs.V, sc, f.bs.P};
    if ((st = zgemm(g, PTN_FP64, PTN_T_C128, PTN_T_C128, PTN_T_C128, nullptr, 0, s))) return st;
    nparts = 1;
  }
  k_qr_reduce<<<dim3((unsigned)((nc + 7) / 8), (unsigned)f.batch), 256, 0, s>>>(
      nbp, nc, nparts, f.P, Tp, adjoint, f.Z, f.bs);
  PTN_LAUNCH_CHECK();
  // C += V Z
  ZGemm g = {mr, nc, nbp, V, 1, m, 0, f.Z, nc, 1, 0, Cs, 1, ldc, 1, f.batch, f.bs.V, f.bs.Z, sc};
  return zgemm(g, PTN_FP64, PTN_T_C128, PTN_T_C128, PTN_T_C128, nullptr, 0, s);
}

// The panel j0 .. pe-1 of at most 2048 rows. One workgroup holds a panel of up to
// 256 rows in its registers; beyond, four columns per launch with every column in a
// workgroup of its own (512 rows: 45 us per panel against 66 in one workgroup; the
// sub-panels of 16 and 8 columns that one CU can hold at 1024 and 2048 rows are bound by
// that CU's FP64 and LDS rates: 90 and 200 us per panel against 52 and 63).
constexpr int64_t QR_ONE_ROWS = 256;
template <int R>
static void panel_one(const QrFact& f, int64_t j0, int64_t pe, double2* Tp, hipStream_t s) {
  const int nbp = (int)(pe - j0);
  if (nbp <= 16)   // four columns per wave: half of the products and sums per reflector
    k_qr_panel<R, 4, 4><<<(unsigned)f.batch, 256, 0, s>>>(f.m, j0, nbp, f.W, f.Vf, f.tau, f.rdiag,
                                                         Tp, f.bs);
  else
    k_qr_panel<R, 8, 4><<<(unsigned)f.batch, 256, 0, s>>>(f.m, j0, nbp, f.W, f.Vf, f.tau, f.rdiag,
                                                         Tp, f.bs);
}
template <int R> static void panel_col4(const QrFact& f, int64_t j0, int64_t pe, hipStream_t s) {
  const unsigned B = (unsigned)f.batch;
  for (int64_t j = j0; j < pe; j += 4)
    k_qr_col4<R><<<dim3((unsigned)(pe - j), B), 256, 0, s>>>(
        f.m, j0, j, (int)(pe - j < 4 ? pe - j : 4), f.W, f.Vf, f.tau, f.rdiag, f.G, f.bs);
  k_qr_fixup4<<<B, 256, 0, s>>>(f.m, j0, (int)(pe - j0), f.G, f.W, f.bs);
}
static void panel(const QrFact& f, int64_t j0, int64_t pe, double2* Tp, hipStream_t s) {
  const int64_t rows = f.m - j0;
  if (rows <= 64) panel_one<1>(f, j0, pe, Tp, s);
  else if (rows <= 128) panel_one<2>(f, j0, pe, Tp, s);
  else if (rows <= QR_ONE_ROWS) panel_one<4>(f, j0, pe, Tp, s);
  else if (rows <= 512) panel_col4<2>(f, j0, pe, s);
  else if (rows <= 1024) panel_col4<4>(f, j0, pe, s);
  else panel_col4<8>(f, j0, pe, s);
}

int qr_factor(QrFact& f, const double2* a, int64_t lda, hipStream_t s, int64_t sa) {
  const int64_t m = f.m, n = f.n, k = f.k;
  if (m == 0 || n == 0) return PTN_OK;
  if (f.batch < 1 || f.batch > 65535) return PTN_ERR_ARG;
  const unsigned B = (unsigned)f.batch;
  if (m * n <= QR_IN_MAX) {
    const int64_t nt = (m * n + 63) / 64 * 64;
    k_qr_in<<<B, (unsigned)(nt < 1024 ? nt : 1024), 0, s>>>((int)m, (int)n, a, lda, f.W, sa, f.bs.W,
                                                           f.scl);
  } else {
    k_zero_u64<<<(unsigned)((f.batch + 255) / 256), 256, 0, s>>>(f.batch, f.mxb);
    {
      int64_t nb = (m * n + 255) / 256;
      const int64_t cap = f.batch > 16 ? 16 : 256;   // workgroups per matrix (one atomic each)
      if (nb > cap) nb = cap;
      k_maxabs<<<dim3((unsigned)nb, B), 256, 0, s>>>(m, n, a, lda, sa, f.mxb);
    }
    k_to_colmajor<<<dim3((unsigned)((m * n + 255) / 256), B), 256, 0, s>>>(m, n, a, lda, f.W, sa,
                                                                             f.bs.W, f.mxb, f.scl);
  }
  PTN_LAUNCH_CHECK();
  for (int64_t p = 0; p < f.npan; ++p) {
    const int64_t j0 = p * QR_NB;
    const int64_t pe = (j0 + QR_NB < k) ? j0 + QR_NB : k;
    const int nbp = (int)(pe - j0);
    double2* Tp = f.T + p * QR_NB * QR_NB;
    if (m - j0 <= 2048) {
      panel(f, j0, pe, Tp, s);
    } else {
      int64_t j = j0;
      for (; j + 1 < pe; j += 2) {
        const dim3 g((unsigned)(pe - j), B);
        if (m - j <= 256 * 16)
          k_qr_col2r<16><<<g, 256, 0, s>>>(m, j, f.W, f.Vf, f.tau, f.rdiag, f.rsup, f.bs);
        else
          k_qr_col2<<<g, 256, 0, s>>>(m, j, f.W, f.Vf, f.tau, f.rdiag, f.rsup, f.bs);
      }
      if (j < pe)
        k_qr_col<<<dim3((unsigned)(pe - j), B), 256, 0, s>>>(m, j, f.W, f.Vf, f.tau, f.rdiag, f.bs);
      if (pe - j0 >= 2) k_qr_fixsup<<<dim3(1, B), QR_NB / 2, 0, s>>>(m, j0, pe, f.rsup, f.W, f.bs);
    }
    if (m - j0 > QR_ONE_ROWS) {
      const int64_t np = vtv_parts(m - j0);
      const int64_t rows = ((m - j0 + np - 1) / np + 127) / 128 * 128;
      const int parts = (int)((m - j0 + rows - 1) / rows);
      k_qr_vtv<<<dim3((unsigned)parts, B), 256, 0, s>>>(m, j0, nbp, (int)rows, f.Vf, f.G, f.bs);
      k_qr_tmat<<<B, 256, 0, s>>>(nbp, parts, f.G, f.tau + j0, Tp, f.bs);
    }
    PTN_LAUNCH_CHECK();
    int st;
    if (pe < n && (st = apply_block(f, j0, nbp, Tp, 1, f.W, m, pe, n - pe, s, f.bs.W))) return st;
  }
  return PTN_OK;
}

int qr_apply_q(const QrFact& f, double2* C, int64_t ldc, int64_t nc, bool identity_tail,
               hipStream_t s, int64_t sc) {
  if (nc > f.ncmax) return PTN_ERR_ARG;
  for (int64_t p = f.npan - 1; p >= 0; --p) {
    const int64_t j0 = p * QR_NB;
    const int64_t pe = (j0 + QR_NB < f.k) ? j0 + QR_NB : f.k;
    const int64_t c0 = identity_tail ? j0 : 0;
    int st;
    if ((st = apply_block(f, j0, (int)(pe - j0), f.T + p * QR_NB * QR_NB, 0, C, ldc, c0, nc - c0,
                          s, sc)))
      return st;
  }
  return PTN_OK;
}

// column-major m x k identity columns (one matrix per blockIdx.y, stride m * k)
__global__ void k_q_init(int64_t m, int64_t k, double2* __restrict__ Qc) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= m * k) return;
  Qc += blockIdx.y * m * k;
  int64_t c = t / m, i = t % m;
  Qc[t] = make_double2(i == c ? 1.0 : 0.0, 0.0);
}

// Q (row-major, ldq) from Qc; R (row-major k x n, ldr) from the upper triangle of W
// with the diagonal from rdiag; matrix b of a batch at q + b * sq, r + b * sr
__global__ void k_qr_out(int64_t m, int64_t n, int64_t k, const double2* __restrict__ W,
                         const double2* __restrict__ rdiag, const double2* __restrict__ Qc,
                         double2* __restrict__ q, int64_t ldq, double2* __restrict__ r,
                         int64_t ldr, QrStrides bs, int64_t sq, int64_t sr,
                         const double* __restrict__ scl) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t b = blockIdx.y;
  const double inv = 1.0 / scl[b];   // exact: scl is a power of two
  W += b * bs.W;
  rdiag += b * bs.k;
  Qc += b * m * k;
  q += b * sq;
  r += b * sr;
  if (t < m * k) {
    int64_t i = t / k, c = t % k;
    q[i * ldq + c] = Qc[c * m + i];
  }
  if (t < k * n) {
    int64_t i = t / n, c = t % n;
    const double2 v = (i < c) ? W[c * m + i] : (i == c ? rdiag[i] : make_double2(0.0, 0.0));
    r[i * ldr + c] = make_double2(v.x * inv, v.y * inv);
  }
}

size_t qr_ws_bytes(int64_t m, int64_t n, int64_t batch) {
  int64_t k = m < n ? m : n;
  return al(qr_fact_bytes(m, n, n, batch)) + al((size_t)batch * m * k * 16);
}

// `batch` row-major m x n matrices stacked contiguously (a: lda = n; q: m x k,
// ldq = k; r: k x n, ldr = n) when batch > 1
int qr_run(int64_t m, int64_t n, const void* a, int64_t lda, void* q, int64_t ldq, void* r,
           int64_t ldr, void* ws, size_t ws_bytes, hipStream_t s, int64_t batch) {
  if (m < 0 || n < 0 || lda < n || ldq < (m < n ? m : n) || ldr < n) return PTN_ERR_ARG;
  if (batch < 1 || batch > 65535) return PTN_ERR_ARG;
  if (ws_bytes < qr_ws_bytes(m, n, batch)) return PTN_ERR_WORKSPACE;
  const int64_t k = m < n ? m : n;
  if (m == 0 || n == 0) return PTN_OK;
  QrFact f = qr_fact_layout(m, n, n, ws, batch);
  double2* Qc = (double2*)((char*)ws + al(qr_fact_bytes(m, n, n, batch)));
  int st;
  if ((st = qr_factor(f, (const double2*)a, lda, s, m * lda))) return st;
  const unsigned B = (unsigned)batch;
  k_q_init<<<dim3((unsigned)((m * k + 255) / 256), B), 256, 0, s>>>(m, k, Qc);
  PTN_LAUNCH_CHECK();
  if ((st = qr_apply_q(f, Qc, m, k, true, s, m * k))) return st;
  const int64_t tot = (m * k > k * n) ? m * k : k * n;
  k_qr_out<<<dim3((unsigned)((tot + 255) / 256), B), 256, 0, s>>>(
      m, n, k, f.W, f.rdiag, Qc, (double2*)q, ldq, (double2*)r, ldr, f.bs, m * ldq, k * ldr,
      f.scl);
  PTN_LAUNCH_CHECK();
  return PTN_OK;
}

}  // namespace ptn
