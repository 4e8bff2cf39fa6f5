// Mode mix of the small MPO index pairs (see ops.hip).
#include "common.h"

namespace ptn {

// ---------------------------------------------------------------------------
// Mode mix: Y[l, o, r] = sum_i Wm[o, i] X[l, i, r] for the small MPO index
// pairs (ni, no <= 32); Wm is stored as [o][i] or transposed as [i][o].
//
// HBM-bound at large bonds (reads ni and writes no complex values per (l, r)),
// latency-bound at small ones. A workgroup takes units of up to 64 (l, r) columns: all
// of its threads load the unit's ni x 64 inputs into LDS, every load in flight
// at once (the next unit's while the current one is mixed), and each of its
// four waves then forms every fourth output from there. Most entries of an MPO tensor are
// zero: a bit mask per output lists the others, so a wave (whose lanes share
// the output) runs over the nonzero entries only, in ascending order. Bonds
// shorter than 64 put 2 or 4 rows l side by side in a unit (RC columns each).
// Two-site H_eff mix (20 x 20): D = 64 30.6 -> 4.8 us, D = 1024 complex128 206 -> 109
// us (one thread per column held its inputs in registers and walked all
// outputs in turn before).
constexpr int MIX_MAX = 32;

// blockIdx.y selects the problem of a batch (strides in complex elements)
template <typename TX, typename TY, typename A, int CAP>
__global__ __launch_bounds__(256) void mode_mix_kernel(int64_t nl, int ni, int no, int64_t nr,
                                                       int rc_log, int nunits,
                                                       const double2* __restrict__ wm, int wtrans,
                                                       const TX* __restrict__ x,
                                                       TY* __restrict__ y, int64_t bw,
                                                       int64_t bx, int64_t by,
                                                       const int* __restrict__ skip,
                                                       int64_t skip_stride) {
  typedef typename cplx_of<A>::type C2;
  constexpr int NP = CAP / 4;                  // inputs per thread and unit
  __shared__ C2 W[CAP * MIX_MAX];
  __shared__ unsigned int nz[MIX_MAX];
  __shared__ C2 X[CAP][64];
  if (skip && skip[blockIdx.y * skip_stride]) return;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  wm += blockIdx.y * bw;
  x += blockIdx.y * bx;
  y += blockIdx.y * by;
  const int rc = 1 << rc_log;
  const int chunks = (int)((nr + rc - 1) >> rc_log);
  // the column (l, r) of this lane in a unit
  auto column = [&](int u, int64_t& l, int64_t& r) -> bool {
    const int row = u / chunks;
    l = (int64_t)row * (64 >> rc_log) + (lane >> rc_log);
    r = (int64_t)(u - row * chunks) * rc + (lane & (rc - 1));
    return l < nl && r < nr;
  };
  C2 pre[NP];
  auto load = [&](int u) {
    int64_t l, r;
    const bool in = column(u, l, r);
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const int i = wave + 4 * k;
      pre[k] = C2{0, 0};
      if (in && i < ni) load_c<A>(x + (l * ni + i) * nr + r, pre[k].x, pre[k].y);
    }
  };
  int u = blockIdx.x;
  load(u);
  if (t < no) nz[t] = 0;
  __syncthreads();
  for (int e = t; e < ni * no; e += 256) {
    const int o = e / ni, i = e - o * ni;
    const double2 w = wm[wtrans ? i * no + o : e];
    W[e] = C2{(A)w.x, (A)w.y};
    if (w.x != 0.0 || w.y != 0.0) atomicOr(&nz[o], 1u << i);
  }
  for (; u < nunits; u += gridDim.x) {
    __syncthreads();   // the previous unit has been mixed
#pragma unroll
    for (int k = 0; k < NP; ++k)
      if (wave + 4 * k < ni) X[wave + 4 * k][lane] = pre[k];
    __syncthreads();
    if (u + gridDim.x < nunits) load(u + gridDim.x);
    int64_t l, r;
    const bool in = column(u, l, r);
    for (int o = wave; o < no; o += 4) {
      A yr = 0, yi = 0;
      for (unsigned int m = __builtin_amdgcn_readfirstlane(nz[o]); m; m &= m - 1) {
        const int i = __builtin_ctz(m);
        const C2 w = W[o * ni + i], v = X[i][lane];
        yr += w.x * v.x - w.y * v.y;
        yi += w.x * v.y + w.y * v.x;
      }
      if (in) store_c(y + (l * no + o) * nr + r, yr, yi);
    }
  }
}

template <int CAP>
static void mix_launch(dim3 grid, int64_t nl, int ni, int no, int64_t nr, int rc_log,
                       int nunits, const void* wm, int wt, const void* x, int tx, void* y,
                       int ty, int64_t bw, int64_t bx, int64_t by, const SkipFlag& sk,
                       hipStream_t s) {
  if (tx == PTN_T_C128 && ty == PTN_T_C128)
    mode_mix_kernel<double2, double2, double, CAP><<<grid, 256, 0, s>>>(
        nl, ni, no, nr, rc_log, nunits, (const double2*)wm, wt, (const double2*)x, (double2*)y, bw,
        bx, by, sk.p, sk.stride);
  else if (tx == PTN_T_C64 && ty == PTN_T_C64)
    mode_mix_kernel<float2, float2, float, CAP><<<grid, 256, 0, s>>>(
        nl, ni, no, nr, rc_log, nunits, (const double2*)wm, wt, (const float2*)x, (float2*)y, bw,
        bx, by, sk.p, sk.stride);
  else if (tx == PTN_T_C128 && ty == PTN_T_C64)
    mode_mix_kernel<double2, float2, double, CAP><<<grid, 256, 0, s>>>(
        nl, ni, no, nr, rc_log, nunits, (const double2*)wm, wt, (const double2*)x, (float2*)y, bw,
        bx, by, sk.p, sk.stride);
  else
    mode_mix_kernel<float2, double2, double, CAP><<<grid, 256, 0, s>>>(
        nl, ni, no, nr, rc_log, nunits, (const double2*)wm, wt, (const float2*)x, (double2*)y, bw,
        bx, by, sk.p, sk.stride);
}

int mode_mix(int64_t nl, int64_t ni, int64_t no, int64_t nr, const void* wm, const void* x, int tx,
             void* y, int ty, hipStream_t s, int64_t batch, int64_t bw, bool wtrans) {
  if (ni > MIX_MAX || no > MIX_MAX || ni < 1 || no < 1) return PTN_ERR_UNSUPPORTED;
  if (nl == 0 || nr == 0 || batch == 0) return PTN_OK;
  if (nl > 65535 || batch > 65535) return PTN_ERR_ARG;
  const int rc_log = nr <= 16 ? 4 : (nr <= 32 ? 5 : 6);
  const int64_t rows = 64 >> rc_log;
  const int64_t nunits = ((nl + rows - 1) / rows) * ((nr + (1 << rc_log) - 1) >> rc_log);
  if (nunits > 0x3fffffff) return PTN_ERR_ARG;
  // beyond the workgroups that fit the chip at once each takes several units
  const int64_t cap = 2048 / batch > 256 ? 2048 / batch : 256;
  const dim3 grid((unsigned)(nunits < cap ? nunits : cap), (unsigned)batch);
  const int64_t bx = nl * ni * nr, by = nl * no * nr;
  const SkipFlag sk = skip_flag();
  if (ni <= 16)
    mix_launch<16>(grid, nl, (int)ni, (int)no, nr, rc_log, (int)nunits, wm, wtrans, x, tx, y, ty, bw,
                   bx, by, sk, s);
  else
    mix_launch<MIX_MAX>(grid, nl, (int)ni, (int)no, nr, rc_log, (int)nunits, wm, wtrans, x, tx,
                        y, ty, bw, bx, by, sk, s);
  PTN_LAUNCH_CHECK();
  return PTN_OK;
}

}  // namespace ptn
