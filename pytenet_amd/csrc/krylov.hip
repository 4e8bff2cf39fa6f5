// Device-resident Lanczos for the local TDVP/DMRG problems.
//
// Follows pytenet/krylov.py:12-57 (plain three-term recurrence, no
// reorthogonalisation, breakdown when beta_j < 100*n*eps), krylov.py:142-150
// (eigendecomposition of the tridiagonal matrix) and krylov.py:110-136
// (Ritz vector / Krylov exponential). All scalars (alpha, beta, norms, the
// tridiagonal eigensystem and the combination coefficients) live in device
// memory and are FP64, so a whole local solve is enqueued without a host
// round trip. A breakdown or a non-finite value stops the recurrence through a
// flag that later kernels read; the host reads the status words afterwards.
#include <float.h>
#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>
#include <unordered_map>
#include "common.h"
#include "ops.h"
#include "wave.h"

namespace ptn {

constexpr int LZ_MAX = 64;        // largest supported numiter
constexpr int RED_BLOCKS = 512;   // largest reduction width (partial sums per reduction)

struct LzState {
  double alpha[LZ_MAX];
  double beta[LZ_MAX];
  double coef_re[LZ_MAX];
  double coef_im[LZ_MAX];
  double nrm0;
  double energy;
  int nvalid;      // Lanczos vectors in use
  int breakdown;   // j + 1 of a beta breakdown, 0 if none
  int nonfinite;   // a norm / inner product was not finite
  int zero_start;  // the start vector had norm zero
  int stopped;     // recurrence stopped (breakdown, non-finite or zero start)
  int noconv;      // tridiagonal QL iteration did not converge
};

// Batched form: blockIdx.y selects the problem of a batch; vector arrays are
// stacked with a per-problem stride, LzState and partial-sum arrays are
// indexed by problem. `rb` partial sums per reduction (rb = min(512,
// ceil(n / 256)), a function of n only, so every sum has a fixed order).

// sum over the workgroup (up to 16 waves) in a fixed order, in every thread: the sums of
// each wave's rows of 16 lanes through LDS, then lane l of a row adds those of wave l. red
// is not written again until the caller's next barrier after it.
// Of the first `waves` waves; the others only take part in the barrier (result 0).
__device__ __forceinline__ double wg_sum(double v, double (&red)[16][4], int waves) {
  const int t = threadIdx.x, w = t & 15;
  const bool on = t >> 6 < waves;
  if (on) {
    v = row_sum(v);
    if (w == 0) red[t >> 6][(t >> 4) & 3] = v;
  }
  lds_barrier();
  if (!on) return 0.0;
  const double s = (red[w][0] + red[w][1]) + (red[w][2] + red[w][3]);
  return row_sum(w < waves ? s : 0.0);
}
__device__ __forceinline__ double wg_sum(double v, double (&red)[16][4]) {
  return wg_sum(v, red, (int)(blockDim.x >> 6));
}

// (the three vector kernels at n = 16384 with sums by halving in LDS 2.9 + 4.3 + 3.9 us, with
// wg_sum 2.5 + 3.3 + 3.3)
// sum of the rb partials in a fixed order; every block of a kernel computes the identical
// value (256 threads)
__device__ __forceinline__ double block_sum_partials(const double* __restrict__ part, int rb) {
  __shared__ __align__(16) double red[16][4];
  double v = 0;
  for (int i = threadIdx.x; i < rb; i += 256) v += part[i];
  return wg_sum(v, red);
}

__device__ __forceinline__ void block_store_partial(double v, double* out) {
  __shared__ __align__(16) double red[16][4];
  const double s = wg_sum(v, red);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

__device__ __forceinline__ void state_init(LzState* st, int numiter) {
  const int t = threadIdx.x;
  if (t < LZ_MAX) {
    st->alpha[t] = 0; st->beta[t] = 0; st->coef_re[t] = 0; st->coef_im[t] = 0;
  }
  if (t == 0) {
    st->nrm0 = 0; st->energy = 0; st->nvalid = numiter; st->breakdown = 0;
    st->nonfinite = 0; st->zero_start = 0; st->stopped = 0; st->noconv = 0;
  }
}

__global__ __launch_bounds__(256) void k_sumsq_partial(int64_t n, const double2* __restrict__ x,
                                                       int64_t xs, double* __restrict__ part,
                                                       int rb, LzState* st, int numiter) {
  if (blockIdx.x == 0) state_init(st + blockIdx.y, numiter);
  x += blockIdx.y * xs;
  part += blockIdx.y * rb;
  double s = 0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)rb * 256) {
    double2 v = x[i];
    s += v.x * v.x + v.y * v.y;
  }
  block_store_partial(s, part);
}

// Re <w, v> partials
__global__ __launch_bounds__(256) void k_dot_partial(int64_t n, const double2* __restrict__ w,
                                                     int64_t ws_, const double2* __restrict__ v,
                                                     int64_t vs, double* __restrict__ part,
                                                     int rb) {
  w += blockIdx.y * ws_;
  v += blockIdx.y * vs;
  part += blockIdx.y * rb;
  double s = 0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)rb * 256) {
    double2 a = w[i], b = v[i];
    s += a.x * b.x + a.y * b.y;
  }
  block_store_partial(s, part);
}

// v0 = x / |x|  (krylov.py:29-31)
__global__ __launch_bounds__(256) void k_start(int64_t n, const double2* __restrict__ x,
                                               int64_t xs, double2* __restrict__ v0, int64_t vs,
                                               const double* __restrict__ part, int rb,
                                               LzState* st) {
  x += blockIdx.y * xs;
  v0 += blockIdx.y * vs;
  part += blockIdx.y * rb;
  st += blockIdx.y;
  double nrm = sqrt(block_sum_partials(part, rb));
  bool bad = !(nrm > 0.0) || !isfinite(nrm);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->nrm0 = nrm;
    if (bad) {
      if (nrm == 0.0) st->zero_start = 1; else st->nonfinite = 1;
      st->stopped = 1;
      st->nvalid = 0;
    }
  }
  if (bad) return;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    double2 a = x[i];
    v0[i] = make_double2(a.x / nrm, a.y / nrm);
  }
}

// alpha_j = Re <w, v_j>;  w -= alpha_j v_j + beta_{j-1} v_{j-1};  partials of |w|^2
__global__ __launch_bounds__(256) void k_alpha_update(int64_t n, double2* __restrict__ w,
                                                      int64_t ws_,
                                                      const double2* __restrict__ vj,
                                                      const double2* __restrict__ vjm1,
                                                      int64_t vs, int j,
                                                      const double* __restrict__ part_in,
                                                      double* __restrict__ part_out, int rb,
                                                      LzState* st) {
  st += blockIdx.y;
  if (st->stopped) return;
  w += blockIdx.y * ws_;
  vj += blockIdx.y * vs;
  vjm1 += blockIdx.y * vs;
  part_in += blockIdx.y * rb;
  part_out += blockIdx.y * rb;
  const double a = block_sum_partials(part_in, rb);
  if (!isfinite(a)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      st->nonfinite = 1; st->stopped = 1; st->nvalid = j + 1; st->alpha[j] = a;
    }
    return;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) st->alpha[j] = a;
  const double b = (j > 0) ? st->beta[j - 1] : 0.0;
  double s = 0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)rb * 256) {
    double2 x = w[i], v = vj[i];
    double tr = a * v.x, ti = a * v.y;
    if (j > 0) {
      double2 u = vjm1[i];
      tr += b * u.x; ti += b * u.y;
    }
    x.x -= tr; x.y -= ti;
    w[i] = x;
    s += x.x * x.x + x.y * x.y;
  }
  block_store_partial(s, part_out);
}

// beta_j = |w|; breakdown test; v_{j+1} = w / beta_j. The test is the
// reference's absolute one (beta_j < 100 n eps) and, for matvecs in reduced
// precision (rel > 0), also beta_j < rel |A v_j| with |A v_j| =
// sqrt(alpha_j^2 + beta_{j-1}^2 + beta_j^2): a residual below the rounding
// noise of a complex64 / split-bf16 matvec is that noise, not a new Krylov
// direction (a start vector in an invariant subspace otherwise continues with
// normalised noise).
__global__ __launch_bounds__(256) void k_beta_next(int64_t n, const double2* __restrict__ w,
                                                   int64_t ws_, double2* __restrict__ vnext,
                                                   int64_t vs, int j,
                                                   const double* __restrict__ part_in, int rb,
                                                   double thresh, double rel, LzState* st) {
  st += blockIdx.y;
  if (st->stopped) return;
  w += blockIdx.y * ws_;
  vnext += blockIdx.y * vs;
  part_in += blockIdx.y * rb;
  const double b = sqrt(block_sum_partials(part_in, rb));
  const bool nf = !isfinite(b);
  const double a = st->alpha[j], bm = j > 0 ? st->beta[j - 1] : 0.0;
  const double thr = fmax(thresh, rel * sqrt(a * a + bm * bm + b * b));
  const bool brk = !nf && (b < thr);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (nf) { st->nonfinite = 1; st->stopped = 1; st->nvalid = j + 1; }
    else if (brk) { st->breakdown = j + 1; st->stopped = 1; st->nvalid = j + 1; }
    else st->beta[j] = b;
  }
  if (nf || brk) return;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    double2 x = w[i];
    vnext[i] = make_double2(x.x / b, x.y / b);
  }
}

// Short vectors: one workgroup per problem keeps its part of the vectors in registers
// and does all of a step at once, R elements per thread (n <= 1024 R). Such a step is bound
// by launches and by the latency of dependent loads and sums. A Lanczos step (inner product,
// update, normalisation) as three launches of 256-thread workgroups and as one: n = 1024 2.7 + 3.9
// + 3.5 -> 4.5 us, 4096 -> 6.5 us, 8192 10.4 -> 11.0 us with two launches and their gaps
// fewer; at 16384 one CU's bandwidth would cost more (the registers spill: 45 us).
constexpr int SHORT_T = 1024;     // largest workgroup
constexpr int64_t SHORT_MAX = 8 * SHORT_T;

// x / b from inv = 1 / b with one correction (b a normal number)
__device__ __forceinline__ double div_by(double x, double b, double inv) {
  const double q = x * inv;
  return fma(fma(-q, b, x), inv, q);
}

// state, norm of the start vector and v0 = x / |x|  (krylov.py:29-31)
template <int R>
__global__ __launch_bounds__(SHORT_T) void k_lz_start(int n, const double2* __restrict__ x,
                                                      double2* __restrict__ v0, LzState* st,
                                                      int numiter) {
  __shared__ __align__(16) double red[16][4];
  x += (int64_t)blockIdx.x * n;
  v0 += (int64_t)blockIdx.x * n;
  st += blockIdx.x;
  const int nt = blockDim.x;
  double2 a[R];
  double s = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = threadIdx.x + r * nt;
    a[r] = i < n ? x[i] : make_double2(0.0, 0.0);
  }
#pragma unroll
  for (int r = 0; r < R; ++r) s += a[r].x * a[r].x + a[r].y * a[r].y;
  state_init(st, numiter);
  const double nrm = sqrt(wg_sum(s, red));
  const bool bad = !(nrm > 0.0) || !isfinite(nrm);
  if (threadIdx.x == 0) {
    st->nrm0 = nrm;
    if (bad) {
      if (nrm == 0.0) st->zero_start = 1; else st->nonfinite = 1;
      st->stopped = 1;
      st->nvalid = 0;
    }
  }
  if (bad) return;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = threadIdx.x + r * nt;
    if (i < n) v0[i] = make_double2(a[r].x / nrm, a[r].y / nrm);
  }
}

// alpha_j, the update of w, beta_j with the breakdown test and v_{j+1} = w / beta_j (the
// formulas of k_dot_partial, k_alpha_update and k_beta_next); w is only read
template <int R>
__global__ __launch_bounds__(SHORT_T) void k_lz_step(int n, const double2* __restrict__ w,
                                                     const double2* __restrict__ vj,
                                                     const double2* __restrict__ vjm1,
                                                     double2* __restrict__ vnext, int j,
                                                     double thresh, double rel, LzState* st) {
  __shared__ __align__(16) double red[2][16][4];
  st += blockIdx.x;
  if (st->stopped) return;
  const int64_t o = (int64_t)blockIdx.x * n;
  w += o;
  vj += o;
  vjm1 += o;
  vnext += o;
  const int nt = blockDim.x;
  const double2 zero = make_double2(0.0, 0.0);
  constexpr bool KEEP = R <= 4;   // v_j and v_{j-1} stay in registers from the first read on
  double2 x[R], v[KEEP ? R : 1], u[KEEP ? R : 1];
  double s = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = threadIdx.x + r * nt;
    x[r] = i < n ? w[i] : zero;
    if constexpr (KEEP) {
      v[r] = i < n ? vj[i] : zero;
      u[r] = j > 0 && i < n ? vjm1[i] : zero;
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = threadIdx.x + r * nt;
    const double2 b = KEEP ? v[KEEP ? r : 0] : (i < n ? vj[i] : zero);
    s += x[r].x * b.x + x[r].y * b.y;
    if (!KEEP && (r & 3) == 3) __builtin_amdgcn_sched_barrier(0);   // loads of four at a time
  }
  const double b0 = j > 0 ? st->beta[j - 1] : 0.0;
  const double a = wg_sum(s, red[0]);
  if (threadIdx.x == 0) st->alpha[j] = a;
  if (!isfinite(a)) {
    if (threadIdx.x == 0) { st->nonfinite = 1; st->stopped = 1; st->nvalid = j + 1; }
    return;
  }
  s = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = threadIdx.x + r * nt;
    const double2 vr = KEEP ? v[KEEP ? r : 0] : (i < n ? vj[i] : zero);
    double tr = a * vr.x, ti = a * vr.y;
    if (j > 0) {
      const double2 ur = KEEP ? u[KEEP ? r : 0] : (i < n ? vjm1[i] : zero);
      tr += b0 * ur.x;
      ti += b0 * ur.y;
    }
    x[r].x -= tr;
    x[r].y -= ti;
    s += x[r].x * x[r].x + x[r].y * x[r].y;
    if (!KEEP && (r & 3) == 3) __builtin_amdgcn_sched_barrier(0);
  }
  const double b = sqrt(wg_sum(s, red[1]));
  const bool nf = !isfinite(b);
  const bool brk = !nf && b < fmax(thresh, rel * sqrt(a * a + b0 * b0 + b * b));
  if (threadIdx.x == 0) {
    if (nf) { st->nonfinite = 1; st->stopped = 1; st->nvalid = j + 1; }
    else if (brk) { st->breakdown = j + 1; st->stopped = 1; st->nvalid = j + 1; }
    else st->beta[j] = b;
  }
  if (nf || brk) return;
  const double inv = 1.0 / b;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = threadIdx.x + r * nt;
    if (i < n) vnext[i] = make_double2(div_by(x[r].x, b, inv), div_by(x[r].y, b, inv));
  }
}

// the value of the next (UP) or the previous lane of the wave, zero beyond its ends
template <bool UP> __device__ __forceinline__ double lane_shift(double v) {
  constexpr int CTRL = UP ? 0x130 : 0x138;   // wave shift left / right by one lane
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double wave_max(double v) {
  v = fmax(v, dpp_rot<0x128>(v));
  v = fmax(v, dpp_rot<0x124>(v));
  v = fmax(v, dpp_rot<0x122>(v));
  v = fmax(v, dpp_rot<0x121>(v));
  return fmax(fmax(lane_value(v, 0), lane_value(v, 16)),
              fmax(lane_value(v, 32), lane_value(v, 48)));
}

// Coefficients of the Krylov vectors from the tridiagonal matrix (alpha, beta) of n
// rows, by one wave (lane k holds row k in registers and returns coefficient k):
//   mode 0 (expm):  c = |v| exp(dt T) e_1                              (krylov.py:132-136)
//   mode 1 (eigh):  c = the eigenvector of the lowest eigenvalue, its energy (krylov.py:116-119)
// The exponential is applied to e_1 by Taylor polynomials of degree 18 in Horner's form, in
// steps of |dt| rho <= 1 with T shifted to the centre of its Gershgorin interval of radius rho
// (the remainder is below 2^-56): a step is 18 products with a tridiagonal matrix, neighbours
// read across the lanes. Up to 16 steps; beyond them, and for mode 1, the
// eigendecomposition below. Error against 50 digits, norm of the result = 1, |dt| rho =
// 0.01 .. 16, imaginary, real and complex dt: 3e-17 .. 9e-16 in the median, largest
// 3.2e-15; from the eigendecomposition (LAPACK) 4e-16 .. 6e-15 and 2.4e-13.
// The last kernel of a solve at n = 10 takes 4 - 6 us with it.
//
// Eigendecomposition by the implicit QL method with Wilkinson shifts: every lane runs
// the same scalar recurrence on values read as scalars, and lane k applies the plane rotations
// to row k of the eigenvector matrix (Z, rows of ldz doubles in LDS). The chain of
// dependent operations of the rotations (about 1.7 n sweeps of n / 2) sets its time:
// r = sqrt(f^2 + g^2), f / r and g / r come from one reciprocal square root (hypot where
// the squares leave the normal range): 25 - 38 us at n = 8 - 10 (40 - 58 with hypot and divisions
// in every rotation and the matrix's diagonals in LDS).
constexpr double TAYLOR_MAX_STEPS = 16.0;
__device__ __forceinline__ bool tridiag_coefs(int n, const double* alpha, const double* beta,
                                              double* Z, int ldz, int mode, double nrm,
                                              double dt_re, double dt_im, double& cr, double& ci,
                                              double& energy) {
  const int lane = threadIdx.x & 63;
  double d = lane < n ? alpha[lane] : 0.0;
  double e = lane < n - 1 ? beta[lane] : 0.0;
  cr = ci = 0.0;
  if (mode == 0) {
    const double em = lane_shift<false>(e);          // coupling to the previous row
    const double off = fabs(e) + fabs(em);
    const double hi = wave_max(lane < n ? d + off : -INFINITY);
    const double lo = -wave_max(lane < n ? off - d : -INFINITY);
    const double mid = 0.5 * (lo + hi), rho = 0.5 * (hi - lo);
    const double steps = fmax(ceil(rho * hypot(dt_re, dt_im)), 1.0);
    if (steps <= TAYLOR_MAX_STEPS) {
      const double zr = dt_re / steps, zi = dt_im / steps, dc = d - mid;
      double x = lane == 0 ? 1.0 : 0.0, y = 0.0;
      for (int q = (int)steps; q > 0; --q) {
        const double x0 = x, y0 = y;
#pragma unroll
        for (int k = 18; k > 0; --k) {
          const double kr = zr * (1.0 / k), ki = zi * (1.0 / k);
          const double tx = fma(dc, x, fma(e, lane_shift<true>(x), em * lane_shift<false>(x)));
          const double ty = fma(dc, y, fma(e, lane_shift<true>(y), em * lane_shift<false>(y)));
          x = fma(kr, tx, fma(-ki, ty, x0));
          y = fma(kr, ty, fma(ki, tx, y0));
        }
      }
      const double mag = nrm * exp(dt_re * mid), ph = dt_im * mid;
      const double er = mag * cos(ph), ei = mag * sin(ph);
      cr = er * x - ei * y;
      ci = er * y + ei * x;
      return true;
    }
  }
  double* zrow = Z + (lane < n ? lane : 0) * ldz;
  if (lane < n)
    for (int k = 0; k < n; ++k) zrow[k] = lane == k ? 1.0 : 0.0;
  bool conv = true;
  for (int l = 0; l < n; ++l) {
    int iter = 0;
    for (;;) {
      const double dn = lane_shift<true>(d);   // by all lanes: a lane that is off reads as zero
      const bool tiny = lane >= l && lane < n - 1 && fabs(e) <= DBL_EPSILON * (fabs(d) + fabs(dn));
      const unsigned long long at = __ballot(tiny);
      const int m = at ? __ffsll(at) - 1 : n - 1;
      if (m == l) break;
      if (++iter > 100) { conv = false; break; }
      // shift from the leading 2 x 2 block of the unreduced part
      const double dl = lane_value(d, l), el = lane_value(e, l);
      double g = (lane_value(d, l + 1) - dl) / (2.0 * el);
      double r = fabs(g) < 1e150 ? sqrt(fma(g, g, 1.0)) : fabs(g);
      g = lane_value(d, m) - dl + el / (g + copysign(r, g));
      double s = 1.0, c = 1.0, p = 0.0;
      double dh = lane_value(d, m);    // d[i + 1]
      double zh = zrow[m];             // Z[.][i + 1]
      bool split = false;
      int i = m - 1;
      for (; i >= l; --i) {
        const double ei = lane_value(e, i), di = lane_value(d, i), z0 = zrow[i];
        const double f = s * ei;
        const double b = c * ei;
        const double h = fma(f, f, g * g);
        if (h > 1e-280 && h < 1e280) {
          const double ri = rsq_full(h);
          r = h * ri;
          s = f * ri;
          c = g * ri;
        } else {
          r = hypot(f, g);
          if (r == 0.0) {
            if (lane == i + 1) { d = dh - p; e = 0.0; }
            if (lane == m) e = 0.0;
            split = true;
            break;
          }
          s = f / r;
          c = g / r;
        }
        if (lane == i + 1) e = r;
        g = dh - p;
        const double t = fma(di - g, s, 2.0 * c * b);
        p = s * t;
        if (lane == i + 1) d = g + p;
        g = fma(c, t, -b);
        zrow[i + 1] = s * z0 + c * zh;
        zh = c * z0 - s * zh;
        dh = di;
      }
      zrow[i + 1] = zh;
      if (split) continue;
      if (lane == l) { d -= p; e = g; }
      if (lane == m) e = 0.0;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
  if (mode == 0) {
    // |v| * exp(dt * lambda_j) * U[0, j] in lane j
    const double mag = nrm * exp(dt_re * d), ph = dt_im * d;
    const double z = lane < n ? Z[lane] : 0.0;
    const double tr = mag * cos(ph) * z, ti = mag * sin(ph) * z;
    for (int j = 0; j < n; ++j) {
      const double u = zrow[j];
      cr = fma(u, lane_value(tr, j), cr);
      ci = fma(u, lane_value(ti, j), ci);
    }
  } else {
    int k = 0;
    energy = lane_value(d, 0);
    for (int j = 1; j < n; ++j) {
      const double dj = lane_value(d, j);
      if (dj < energy) { energy = dj; k = j; }
    }
    cr = zrow[k];
  }
  return conv;
}

// The end of a solve, one workgroup per problem: the last alpha (krylov.py:54-56; from
// the rb partial sums, or for short vectors, rb = 0, straight from w and v_j), the
// coefficients and the exported scalars.
__global__ __launch_bounds__(SHORT_T) void k_lz_tail(int n, const double2* __restrict__ w,
                                                     const double2* __restrict__ vj, int j,
                                                     const double* __restrict__ part, int rb,
                                                     LzState* st, int mode, double dt_re,
                                                     double dt_im, int32_t* info,
                                                     double* alpha_beta, double* energy) {
  __shared__ __align__(16) double red[16][4], Z[LZ_MAX * (LZ_MAX + 1)];
  const int b = blockIdx.x, t = threadIdx.x;
  st += b;
  const int numiter = j + 1;
  const bool go = !st->stopped;
  double a = 0;
  if (go) {
    if (rb) {
      for (int i = t; i < rb; i += blockDim.x) a += part[(int64_t)b * rb + i];
    } else {
      const int64_t o = (int64_t)b * n;
#pragma unroll 4
      for (int i = t; i < n; i += blockDim.x) {
        const double2 x = w[o + i], v = vj[o + i];
        a += x.x * v.x + x.y * v.y;
      }
    }
    a = wg_sum(a, red);
  }
  if (t >= 64) return;
  if (go && t == 0) {
    st->alpha[j] = a;
    if (!isfinite(a)) st->nonfinite = 1;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
  const int nv = st->nvalid;
  double en = 0.0;
  bool conv = true;
  if (nv > 0 && !st->nonfinite) {
    double cr, ci;
    conv = tridiag_coefs(nv, st->alpha, st->beta, Z, LZ_MAX + 1, mode, st->nrm0, dt_re, dt_im, cr,
                         ci, en);
    if (t < nv) {
      st->coef_re[t] = cr;
      st->coef_im[t] = ci;
    }
  }
  if (t == 0) {
    st->energy = en;
    st->noconv = !conv;
    if (info) {
      info[4 * b] = nv;
      info[4 * b + 1] = st->breakdown;
      info[4 * b + 2] = st->nonfinite | (conv ? 0 : 2);
      info[4 * b + 3] = st->zero_start;
    }
    if (energy) energy[b] = en;
  }
  if (alpha_beta && t < numiter) {
    double* ab = alpha_beta + (int64_t)2 * numiter * b;
    ab[t] = st->alpha[t];
    ab[numiter + t] = st->beta[t];
  }
}

}  // namespace ptn

#include "krylov_small.h"

namespace ptn {

// out = sum_{j < nvalid} c_j V_j  (krylov.py:118, :136)
// V_j of problem b at V + j * js + b * Vs
__global__ __launch_bounds__(256) void k_combine(int64_t n, const double2* __restrict__ V,
                                                 int64_t js, int64_t Vs,
                                                 const LzState* __restrict__ st,
                                                 double2* __restrict__ out, int64_t os) {
  __shared__ double cr[LZ_MAX], ci[LZ_MAX];
  V += blockIdx.y * Vs;
  out += blockIdx.y * os;
  st += blockIdx.y;
  const int nv = st->nonfinite ? 0 : st->nvalid;
  if (threadIdx.x < LZ_MAX) {
    cr[threadIdx.x] = st->coef_re[threadIdx.x];
    ci[threadIdx.x] = st->coef_im[threadIdx.x];
  }
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    double sr = 0, si = 0;
    for (int j = 0; j < nv; ++j) {
      const double2 v = V[(int64_t)j * js + i];
      sr += cr[j] * v.x - ci[j] * v.y;
      si += cr[j] * v.y + ci[j] * v.x;
    }
    out[i] = make_double2(sr, si);
  }
}

// ---------------------------------------------------------------------------
static inline size_t al(size_t b) { return (b + 255) & ~(size_t)255; }

struct KrylovLayout {
  size_t v, w, part_a, part_b, state, l64, r64, mv, total;
};

static int64_t op_vec_len(const ptn_local_op* op) {
  return op->kind == PTN_OP_HEFF ? op->Dl * op->d * op->Dr : op->Dl * op->Dr;
}

static int red_width(int64_t n) {
  int64_t rb = (n + 255) / 256;
  if (rb > RED_BLOCKS) rb = RED_BLOCKS;
  return rb < 1 ? 1 : (int)rb;
}

// Krylov vectors are stored as [j][problem][n], so that V_j of all problems is
// one contiguous batch for the batched matvec
static KrylovLayout krylov_layout(const ptn_local_op* op, int numiter, int64_t batch) {
  KrylovLayout k;
  const int64_t n = op_vec_len(op);
  const int rb = red_width(n);
  size_t off = 0;
  k.v = off; off += al((size_t)batch * numiter * n * 16);
  k.w = off; off += al((size_t)batch * n * 16);
  k.part_a = off; off += al((size_t)batch * rb * 8);
  k.part_b = off; off += al((size_t)batch * rb * 8);
  k.state = off; off += al((size_t)batch * sizeof(LzState));
  const bool lowp = (op->precision & ~PTN_BLOCK_SPARSE) != PTN_FP64;
  const int64_t nl = op->Dl * op->Ml * op->Dl, nr = op->Dr * op->Mr * op->Dr;
  k.l64 = off; off += lowp ? al((size_t)batch * nl * 8) : 0;
  k.r64 = off; off += lowp ? al((size_t)batch * nr * 8) : 0;
  k.mv = off;
  if (op->kind == PTN_OP_HEFF) {
    Dims D = {op->Dl, op->d, op->Dr, op->Ml, op->Mr};
    off += al(heff_ws_bytes(op->precision, D, batch));
  } else {
    off += al(bond_ws_bytes(op->precision, op->Dl, op->Dr, op->Ml, batch));
  }
  k.total = off;
  return k;
}

size_t krylov_ws_bytes(const ptn_local_op* op, int numiter, int64_t batch) {
  return krylov_layout(op, numiter, batch).total;
}

// `batch` independent local problems of identical shape: l, w, r, v and out
// stacked contiguously along a leading batch axis; info / energy /
// alpha_beta per problem (4, 1, 2 numiter entries)
static int krylov_enqueue(const ptn_local_op* op, int mode, const void* v, double dt_re,
                          double dt_im, int numiter, void* out, double* energy, int32_t* info,
                          double* alpha_beta, void* ws, size_t ws_bytes, hipStream_t s,
                          int64_t batch, const SectorPlan* sp);

// ---------------------------------------------------------------------------
// hipGraph capture of the local solves (off unless ptn_set_graphs turns it on). A
// solve's whole launch sequence (state init, every Lanczos iteration with its
// matvec, the tridiagonal eigensolver, the combination) is captured into a graph on a
// private stream and launched as one graph on the caller's stream. The
// executable graphs are cached per shape bucket (operator kind and shapes,
// precision, numiter, mode, batch, device) and updated in place with the
// new call's pointers (hipGraphExecUpdate; the topology of one bucket never
// changes). Iterations after a breakdown are predicated off on the device
// (the "stopped" word), so one graph serves every outcome. Each bucket keeps a
// ring of GRAPH_RING executables; an executable is updated only after its
// previous launch has completed (an event per slot). Long vectors (MFMA-bound
// matvecs of milliseconds) are launched directly.
// Direct launches are the default: capturing and updating ~60 nodes costs the host more
// than launching them (two-site expm at D = 64: 260 us against 272; a two-site
// TDVP step of 12 sites 21.9 ms against 25.1; 24 batched chains 55.5 ms against 58.7).
namespace {
bool g_graphs_on = false;
constexpr int64_t GRAPH_MAX_N = 1 << 20;   // vector length up to which solves are captured
constexpr int GRAPH_RING = 3;
constexpr size_t GRAPH_MAX_BUCKETS = 512;
constexpr int GRAPH_GROUPED = 1 << 20;   // key bit: matvecs through the sector-grouped products
struct GKey {
  int dev, kind, prec, mode, numiter;
  int64_t Dl, d, Dr, Ml, Mr, batch;
  bool operator==(const GKey& o) const {
    return dev == o.dev && kind == o.kind && prec == o.prec && mode == o.mode &&
           numiter == o.numiter && Dl == o.Dl && d == o.d && Dr == o.Dr && Ml == o.Ml &&
           Mr == o.Mr && batch == o.batch;
  }
};
struct GHash {
  size_t operator()(const GKey& k) const {
    size_t h = (size_t)k.dev * 1000003u ^ (size_t)k.kind * 10007u ^ (size_t)k.prec * 101u ^
               (size_t)k.mode * 7u ^ (size_t)k.numiter;
    for (int64_t x : {k.Dl, k.d, k.Dr, k.Ml, k.Mr, k.batch}) h = h * 1315423911u ^ (size_t)x;
    return h;
  }
};
struct GEntry {
  hipGraphExec_t exec[GRAPH_RING] = {};
  hipEvent_t done[GRAPH_RING] = {};
  int next = 0;
};
std::mutex g_gmu;
std::unordered_map<GKey, GEntry, GHash> g_graph_cache;
std::map<int, hipStream_t> g_capture_streams;
int64_t g_graph_launches = 0;

void drop_entry(GEntry& e) {
  for (int i = 0; i < GRAPH_RING; ++i) {
    if (e.done[i]) { (void)hipEventSynchronize(e.done[i]); (void)hipEventDestroy(e.done[i]); }
    if (e.exec[i]) (void)hipGraphExecDestroy(e.exec[i]);
    e.exec[i] = nullptr;
    e.done[i] = nullptr;
  }
}
}  // namespace

bool krylov_graphs(int on) {
  std::lock_guard<std::mutex> lk(g_gmu);
  const bool prev = g_graphs_on;
  if (on >= 0) g_graphs_on = on != 0;
  return prev;
}

int64_t krylov_graph_launches() {
  std::lock_guard<std::mutex> lk(g_gmu);
  return g_graph_launches;
}

int krylov_run(const ptn_local_op* op, int mode, const void* v, double dt_re, double dt_im,
               int numiter, void* out, double* energy, int32_t* info, double* alpha_beta,
               void* ws, size_t ws_bytes, hipStream_t s, int64_t batch) {
  if (!op || numiter < 1 || numiter > LZ_MAX || batch < 1 || batch > 65535) return PTN_ERR_ARG;
  const int64_t n = op->kind == PTN_OP_HEFF ? op->Dl * op->d * op->Dr : op->Dl * op->Dr;
  bool use_graph;
  {
    std::lock_guard<std::mutex> lk(g_gmu);
    use_graph = g_graphs_on && n * batch <= GRAPH_MAX_N;
  }
  hipStreamCaptureStatus cst = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &cst) != hipSuccess) cst = hipStreamCaptureStatusActive;
  if (cst != hipStreamCaptureStatusNone)
    use_graph = false;   // the caller captures (or the query failed): launch into its capture
  // the sector plan (quantum-number blocks) is looked up or built here, outside
  // any capture (building copies synchronously); under the caller's own capture
  // the tile-mask products run. The reference keeps the plan alive until the
  // solve is enqueued.
  SectorPlanRef spr;
  if (batch == 1 && cst == hipStreamCaptureStatusNone) {
    const int e = sector_plan_get(op, SECTORS_HEFF, &spr);
    if (e) return e;
  }
  const SectorPlan* sp = spr.get();
  if (!use_graph)
    return krylov_enqueue(op, mode, v, dt_re, dt_im, numiter, out, energy, info, alpha_beta, ws,
                          ws_bytes, s, batch, sp);
  int dev = 0;
  PTN_HIP_CHECK(hipGetDevice(&dev));
  hipStream_t cap;
  {
    std::lock_guard<std::mutex> lk(g_gmu);
    auto it = g_capture_streams.find(dev);
    if (it == g_capture_streams.end()) {
      hipStream_t ns;
      PTN_HIP_CHECK(hipStreamCreateWithFlags(&ns, hipStreamNonBlocking));
      it = g_capture_streams.emplace(dev, ns).first;
    }
    cap = it->second;
  }
  PTN_HIP_CHECK(hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal));
  const int st = krylov_enqueue(op, mode, v, dt_re, dt_im, numiter, out, energy, info, alpha_beta,
                                ws, ws_bytes, cap, batch, sp);
  hipGraph_t g = nullptr;
  const hipError_t ec = hipStreamEndCapture(cap, &g);
  if (st) {
    if (g) (void)hipGraphDestroy(g);
    return st;
  }
  if (ec != hipSuccess) { ptn_set_last_hip_error(ec); return PTN_ERR_HIP; }
  const GKey key{dev, op->kind, op->precision | (sp ? GRAPH_GROUPED : 0), mode, numiter,
                 op->Dl, op->d, op->Dr, op->Ml, op->Mr, batch};
  std::lock_guard<std::mutex> lk(g_gmu);
  if (g_graph_cache.size() >= GRAPH_MAX_BUCKETS && !g_graph_cache.count(key)) {
    for (auto& kv : g_graph_cache) drop_entry(kv.second);
    g_graph_cache.clear();
  }
  GEntry& E = g_graph_cache[key];
  const int slot = E.next;
  E.next = (slot + 1) % GRAPH_RING;
  hipError_t e = hipSuccess;
  if (E.exec[slot]) {
    // the slot's previous launch must be complete before its parameters change
    if ((e = hipEventSynchronize(E.done[slot])) != hipSuccess) {
      (void)hipGraphDestroy(g);
      ptn_set_last_hip_error(e);
      return PTN_ERR_HIP;
    }
    hipGraphNode_t err_node = nullptr;
    hipGraphExecUpdateResult res;
    if (hipGraphExecUpdate(E.exec[slot], g, &err_node, &res) != hipSuccess) {
      (void)hipGetLastError();
      (void)hipGraphExecDestroy(E.exec[slot]);
      E.exec[slot] = nullptr;
    }
  }
  if (!E.exec[slot] && (e = hipGraphInstantiate(&E.exec[slot], g, nullptr, nullptr, 0)) != hipSuccess) {
    E.exec[slot] = nullptr;
    (void)hipGraphDestroy(g);
    ptn_set_last_hip_error(e);
    return PTN_ERR_HIP;
  }
  (void)hipGraphDestroy(g);
  if (!E.done[slot] && (e = hipEventCreateWithFlags(&E.done[slot], hipEventDisableTiming)) != hipSuccess) {
    ptn_set_last_hip_error(e);
    return PTN_ERR_HIP;
  }
  if ((e = hipGraphLaunch(E.exec[slot], s)) != hipSuccess || (e = hipEventRecord(E.done[slot], s)) != hipSuccess) {
    ptn_set_last_hip_error(e);
    return PTN_ERR_HIP;
  }
  ++g_graph_launches;
  return PTN_OK;
}

// f with the elements per thread of the short-vector kernels as a constant
template <typename F> static void short_r(int64_t n, F f) {
  if (n <= SHORT_T) f(std::integral_constant<int, 1>());
  else if (n <= 2 * SHORT_T) f(std::integral_constant<int, 2>());
  else if (n <= 4 * SHORT_T) f(std::integral_constant<int, 4>());
  else f(std::integral_constant<int, 8>());
}

static int krylov_enqueue(const ptn_local_op* op, int mode, const void* v, double dt_re,
                          double dt_im, int numiter, void* out, double* energy, int32_t* info,
                          double* alpha_beta, void* ws, size_t ws_bytes, hipStream_t s,
                          int64_t batch, const SectorPlan* sp) {
  if (!op || numiter < 1 || numiter > LZ_MAX || batch < 1 || batch > 65535) return PTN_ERR_ARG;
  if (op->kind != PTN_OP_HEFF && op->kind != PTN_OP_BOND) return PTN_ERR_ARG;
  const int bprec = op->precision & ~PTN_BLOCK_SPARSE;
  if (bprec != PTN_FP64 && bprec != PTN_FP32 && bprec != PTN_BF16X3 && bprec != PTN_BF16X6)
    return PTN_ERR_UNSUPPORTED;
  if (op->Dl <= 0 || op->Dr <= 0 || op->Ml <= 0 || op->Mr <= 0) return PTN_ERR_ARG;
  if (op->kind == PTN_OP_HEFF && (op->d <= 0 || !op->w)) return PTN_ERR_ARG;
  if (op->kind == PTN_OP_BOND && op->Ml != op->Mr) return PTN_ERR_ARG;
  const KrylovLayout K = krylov_layout(op, numiter, batch);
  if (ws_bytes < K.total) return PTN_ERR_WORKSPACE;
  char* base = (char*)ws;
  double2* V = (double2*)(base + K.v);
  double2* w = (double2*)(base + K.w);
  double* pa = (double*)(base + K.part_a);
  double* pb = (double*)(base + K.part_b);
  LzState* st = (LzState*)(base + K.state);
  void* mvws = base + K.mv;
  const size_t mvbytes = K.total - K.mv;
  const int64_t n = op_vec_len(op);
  const int rb = red_width(n);
  const int64_t js = batch * n;   // stride between V_j and V_{j+1}
  const double thresh = 100.0 * (double)n * DBL_EPSILON;
  // relative breakdown level of reduced-precision matvecs (0: FP64, the reference's rule;
  // the three-term split has the accuracy of an FP32 product)
  const double rel = (bprec == PTN_FP32 || bprec == PTN_BF16X6)
                         ? 128.0 * FLT_EPSILON
                         : (bprec == PTN_BF16X3 ? 1.0 / 4096 : 0.0);

  // (in a batch, a problem's output must not lie over what another workgroup still reads)
  auto apart = [&](const void* q, int64_t elems) {
    const char *o = (const char*)out, *x = (const char*)q;
    return !q || x + batch * elems * 16 <= o || o + batch * n * 16 <= x;
  };
  LzSmall sm;
  if (small_plan(op, numiter, batch, &sm) &&
      (batch == 1 || ((v == out || apart(v, n)) && apart(op->l, op->Dl * op->Ml * op->Dl) &&
                      apart(op->r, op->Dr * op->Mr * op->Dr) &&
                      apart(op->w, op->Ml * op->d * op->d * op->Mr)))) {
    sm.mode = mode;
    sm.thresh = thresh;
    sm.dt_re = dt_re;
    sm.dt_im = dt_im;
    sm.l = (const double2*)op->l;
    sm.w = (const double2*)op->w;
    sm.r = (const double2*)op->r;
    sm.v = (const double2*)v;
    sm.V = V;
    sm.out = (double2*)out;
    sm.js = js;
    sm.info = info;
    sm.alpha_beta = alpha_beta;
    sm.energy = energy;
    small_solve(sm, batch, s);
    PTN_LAUNCH_CHECK();
    return PTN_OK;
  }

  // environment blocks in the matvec's operand precision, converted once per solve
  const void* L = op->l;
  const void* R = op->r;
  int tl = PTN_T_C128, tr = PTN_T_C128;
  int st_;
  if (bprec != PTN_FP64) {
    const int64_t nl = op->Dl * op->Ml * op->Dl, nr = op->Dr * op->Mr * op->Dr;
    if ((st_ = convert_c128_c64(batch * nl, op->l, base + K.l64, s))) return st_;
    if ((st_ = convert_c128_c64(batch * nr, op->r, base + K.r64, s))) return st_;
    L = base + K.l64; R = base + K.r64;
    tl = tr = PTN_T_C64;
  }
  Dims D = {op->Dl, op->d, op->Dr, op->Ml, op->Mr};
  auto matvec = [&](const double2* x, double2* y) -> int {
    if (op->kind == PTN_OP_HEFF && sp && batch == 1)
      return heff_apply_sectors(op->precision, D, sp, L, tl, op->w, R, tr, x, y, mvws, mvbytes, s);
    if (op->kind == PTN_OP_HEFF)
      return heff_apply(op->precision, D, L, tl, op->w, R, tr, x, PTN_T_C128, y, PTN_T_C128,
                        mvws, mvbytes, s, batch);
    return bond_apply(op->precision, op->Dl, op->Dr, op->Ml, L, tl, R, tr, x, PTN_T_C128, y,
                      PTN_T_C128, mvws, mvbytes, s, batch);
  };
  int64_t gblocks = (n + 255) / 256;
  if (gblocks > 2048) gblocks = 2048;
  if (gblocks < 1) gblocks = 1;
  const unsigned B = (unsigned)batch;

  // after a stop (breakdown, non-finite value, zero start) the products of the
  // remaining matvecs of that problem do no work
  static_assert(sizeof(LzState) % sizeof(int) == 0, "LzState stride in ints");
  SkipGuard skip(&st->stopped, (int64_t)(sizeof(LzState) / sizeof(int)));
  const double2* x0 = (const double2*)v;
  const bool shrt = n <= SHORT_MAX;
  const int ni = (int)std::min<int64_t>(n, SHORT_MAX);
  const dim3 nt((unsigned)std::min<int64_t>(SHORT_T, (n + 63) / 64 * 64));
  if (shrt) {
    short_r(n, [&](auto r) { k_lz_start<r.value><<<B, nt, 0, s>>>(ni, x0, V, st, numiter); });
  } else {
    k_sumsq_partial<<<dim3(rb, B), 256, 0, s>>>(n, x0, n, pa, rb, st, numiter);
    k_start<<<dim3((unsigned)gblocks, B), 256, 0, s>>>(n, x0, n, V, n, pa, rb, st);
  }
  PTN_LAUNCH_CHECK();
  for (int j = 0; j < numiter; ++j) {
    double2* vj = V + (int64_t)j * js;
    const double2* vp = j > 0 ? vj - js : vj;
    if ((st_ = matvec(vj, w))) return st_;
    if (!shrt) k_dot_partial<<<dim3(rb, B), 256, 0, s>>>(n, w, n, vj, n, pa, rb);
    if (j == numiter - 1) {
      k_lz_tail<<<B, shrt ? nt : dim3(512), 0, s>>>(ni, w, vj, j, pa, shrt ? 0 : rb, st, mode, dt_re,
                                                    dt_im, info, alpha_beta, energy);
    } else if (shrt) {
      short_r(n, [&](auto r) {
        k_lz_step<r.value><<<B, nt, 0, s>>>(ni, w, vj, vp, vj + js, j, thresh, rel, st);
      });
    } else {
      k_alpha_update<<<dim3(rb, B), 256, 0, s>>>(n, w, n, vj, vp, n, j, pa, pb, rb, st);
      k_beta_next<<<dim3((unsigned)gblocks, B), 256, 0, s>>>(n, w, n, vj + js, n, j, pb, rb,
                                                              thresh, rel, st);
    }
    PTN_LAUNCH_CHECK();
  }
  k_combine<<<dim3((unsigned)gblocks, B), 256, 0, s>>>(n, V, js, n, st, (double2*)out, n);
  PTN_LAUNCH_CHECK();
  return PTN_OK;
}

// ---------------------------------------------------------------------------
// Allocation-free local solve (ptn_krylov_expm_noalloc): the same kernels as
// ptn_krylov_expm, launched directly (no graph), with the workspace in a
// file-scope device array instead of caller or library allocations. Each GPU
// holds its own copy of the array (for the life of the process); its address
// on a device is taken once with hipGetSymbolAddress while that device is
// current and kept per device: the array's name in host code is only a
// host-side stand-in and is never passed to a kernel. Nothing in the
// workspace needs to start at zero (the state block is initialised by the
// first kernel of every solve, every partial sum is written before it is
// read). Calls that overlap on one GPU share the array and race.
__device__ __align__(256) unsigned char scratch[PTN_NOALLOC_SCRATCH_BYTES];

namespace {
std::mutex g_scratch_mu;
std::map<int, void*> g_scratch_ptr;
}  // namespace

static int scratch_address(void** out) {
  int dev = 0;
  PTN_HIP_CHECK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  auto it = g_scratch_ptr.find(dev);
  if (it == g_scratch_ptr.end()) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      ptn_set_last_hip_error(e != hipSuccess ? e : hipErrorInvalidSymbol);
      return PTN_ERR_HIP;
    }
    it = g_scratch_ptr.emplace(dev, p).first;
  }
  *out = it->second;
  return PTN_OK;
}

int krylov_expm_noalloc(const ptn_local_op* op, const void* v, double dt_re, double dt_im,
                        int numiter, void* out, int32_t* info, double* alpha_beta, hipStream_t s) {
  if (!op || numiter < 1 || numiter > LZ_MAX) return PTN_ERR_ARG;
  if (krylov_ws_bytes(op, numiter, 1) > (size_t)PTN_NOALLOC_SCRATCH_BYTES) return PTN_ERR_WORKSPACE;
  void* ws = nullptr;
  int st = scratch_address(&ws);
  if (st) return st;
  NoAllocGuard guard;
  // no sector plan: building one allocates (the tile-mask products run instead)
  return krylov_enqueue(op, 0, v, dt_re, dt_im, numiter, out, nullptr, info, alpha_beta, ws,
                        (size_t)PTN_NOALLOC_SCRATCH_BYTES, s, 1, nullptr);
}

}  // namespace ptn
