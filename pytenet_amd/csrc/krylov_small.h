// A whole local solve of a small problem in one launch, one workgroup per problem
// (included by krylov.hip, whose state and scalar routines it shares).
//
// Near the ends of a chain a matvec is 10^4 - 10^6 flops: its three launches and
// the vector steps' are 3 - 4 us each whatever they compute, ten times over in a solve.
// Here the start vector's norm, every Lanczos step with its matvec, the coefficients
// and the combination run in one workgroup: T1, T2, the current vector and the MPO
// tensor's entries stay in LDS, the products run on wave tiles of 16 x 8
// complex outputs (two FP64 MFMAs per four k) with the environment blocks read from L2, and
// only the Krylov vectors go to memory (read back by the threads that wrote them).
// One CU has 1/256 of the chip's matrix rate (0.28 TFLOP/s) and every phase of a
// matvec waits for LDS and L2, so this pays up to SMALL_FLOP per matvec and one workgroup per
// CU. expm with 10 steps, MPO bond 5, one launch against the launches per step: two sites
// D = 8 168 -> 58 us, 14 193 -> 127; one site D = 16 178 -> 86, 16 x 24 (1.2 MFLOP per
// matvec) 192 -> 123; the two meet near 2 MFLOP.
#include "wave_product.h"

namespace ptn {

constexpr double SMALL_FLOP = 1.6e6;
constexpr int64_t SMALL_CUS = 256;
constexpr int64_t SMALL_N = 2048;        // longest vector
constexpr int SMALL_LDS = 148 * 1024;
constexpr int SMALL_MIX = 32;            // largest row or column count of the MPO matrix (as mode_mix)
constexpr int SMALL_W = 1024;            // largest number of its entries

struct LzSmall {
  int heff, Dl, d, Dr, Ml, Mr, n, numiter, mode;
  SmallProduct g1, g3;                    // T1 = A R, w = L^T T2
  int ld1, ld2, parts;                    // row lengths of T1, T2; parts of the mix's rows
  int o_t1, o_t2, o_w, o_mpo, lds;        // complex offsets in LDS, bytes used
  float rdr;                              // 1 / Dr
  double thresh, dt_re, dt_im;
  const double2 *l, *w, *r, *v;
  double2 *V, *out;
  int64_t js;
  int32_t* info;
  double *alpha_beta, *energy;
};

__global__ __launch_bounds__(SHORT_T) void k_lz_solve(LzSmall g) {
  constexpr int NT = SHORT_T, E = SMALL_N / NT;
  __shared__ __align__(16) double2 lds[SMALL_LDS / 16];
  __shared__ __align__(16) double red[3][16][4];
  __shared__ double al[LZ_MAX], be[LZ_MAX], cre[LZ_MAX], cim[LZ_MAX];
  __shared__ int part_end[SMALL_MIX + 1], used[SMALL_MIX];
  __shared__ short src[SMALL_W], dst[SMALL_W], row[SMALL_W];
  __shared__ int count[SMALL_W / 64];
  __shared__ int conv_s, st[4];
  __shared__ double en_s;
  const int t = threadIdx.x, b = blockIdx.x, n = g.n;
  const double2* L = g.l + (int64_t)b * g.Dl * g.Ml * g.Dl;
  const double2* R = g.r + (int64_t)b * g.Dr * g.Mr * g.Dr;
  double2* V = g.V + (int64_t)b * n;
  double2* v = lds;
  double2 *t1 = lds + g.o_t1, *t2 = lds + g.o_t2, *wv = lds + g.o_w, *mpo = lds + g.o_mpo;
  const int ni = g.d * g.Mr, no = g.Ml * g.d;

  // start vector, its norm, and the MPO matrix with the nonzero inputs of each output row
  double2 x[E], vc[E], vp[E];
  double s = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = t + e * NT;
    x[e] = i < n ? g.v[(int64_t)b * n + i] : make_double2(0.0, 0.0);
    vp[e] = make_double2(0.0, 0.0);
    s += x[e].x * x[e].x + x[e].y * x[e].y;
  }
  if (t < LZ_MAX) al[t] = be[t] = cre[t] = cim[t] = 0.0;
  // the MPO matrix's nonzero entries in the order of (output row, input), counted by ballots
  static_assert(SMALL_W == NT, "one entry per thread");
  double2 we = make_double2(0.0, 0.0);
  unsigned long long has = 0;
  if (g.heff) {
    if (t < no * ni) we = g.w[(int64_t)b * no * ni + t];
    has = __ballot(we.x != 0.0 || we.y != 0.0);
    if ((t & 63) == 0) count[t >> 6] = __popcll(has);
    if (t < no) used[t] = 0;
  }
  const double nrm = sqrt(wg_sum(s, red[0]));
  if (g.heff) {
    int at = 0, total = 0;
#pragma unroll
    for (int q = 0; q < NT / 64; ++q) {
      at += q < t >> 6 ? count[q] : 0;
      total += count[q];
    }
    if (has >> (t & 63) & 1) {
      at += __popcll(has & ((1ull << (t & 63)) - 1));
      const int o = t / ni, k = t - o * ni;
      mpo[at] = we;
      src[at] = (short)(k / g.Mr * g.ld1 + k % g.Mr * g.Dr);
      row[at] = (short)o;
      used[o] = 1;
    }
    __syncthreads();
    // a row's last entry stores it; a row without entries is zero throughout
    for (int c = t; c < total; c += NT) {
      const int o = row[c];
      dst[c] = c + 1 == total || row[c + 1] != o ? (short)(o / g.d * g.ld2 + o % g.d * g.Dr)
                                                 : (short)-1;
    }
    if (t < no && !used[t])
      for (int l = 0; l < g.Dl; ++l)
        for (int r = 0; r < g.Dr; ++r)
          t2[(l * g.Ml + t / g.d) * g.ld2 + t % g.d * g.Dr + r] = make_double2(0.0, 0.0);
    // parts of whole rows with about the same number of entries
    if (t <= g.parts) {
      int c = total * t / g.parts;
      while (c > 0 && c < total && row[c] == row[c - 1]) ++c;
      part_end[t] = c;
    }
  }
  // vectors in use, breakdown step + 1, non-finite value, zero start: uniform through LDS
  const bool bad = !(nrm > 0.0) || !isfinite(nrm);
  if (t == 0) {
    st[0] = bad ? 0 : g.numiter;
    st[1] = 0;
    st[2] = bad && nrm != 0.0;
    st[3] = nrm == 0.0;
  }
  const int waves = min(NT, (n + 63) & ~63) >> 6;   // waves that hold elements
  const bool mine = t >> 6 < waves;
  if (!bad) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = t + e * NT;
      vc[e] = make_double2(x[e].x / nrm, x[e].y / nrm);
      if (i < n) v[i] = V[i] = vc[e];
    }
    __syncthreads();
    double b0 = 0.0;
    for (int j = 0; j < g.numiter; ++j) {
      // T1[(l, s), (m', r')] = A R, T2 = W T1, w = L^T T2
      const auto same = [](int n_) { return n_; };
      const int wcols = g.g3.N;
      const auto out_at = [&](int p, int m_, int n_, int part) {
        return (double*)&wv[p * n + m_ * wcols + n_] + part;
      };
      small_product<false>(g.g1, (const double2*)v, R, same, [&](int, int m_, int n_, int part) {
        return (double*)&t1[m_ * g.ld1 + n_] + part;
      });
      lds_barrier();
      if (g.heff) {
        // a thread takes a unit (l, r') and a part of the rows' entries
        const int units = g.Dl * g.Dr, up = (units + 63) & ~63;
        const int part = g.parts == 1 ? 0 : __builtin_amdgcn_readfirstlane(t) / up;
        if (part < g.parts) {
          const int e0 = part_end[part], e1 = part_end[part + 1];
          for (int u = t - part * up; u < units; u += NT) {
            const int l = (int)(((float)u + 0.5f) * g.rdr), rp = u - l * g.Dr;   // exact
            const double2* in = t1 + l * g.d * g.ld1 + rp;
            double2* to = t2 + l * g.Ml * g.ld2 + rp;
            double yr = 0.0, yi = 0.0;
            for (int e = e0; e < e1; e += 4) {
              double2 c[4], z[4];
              int at[4];
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const int f = min(e + q, e1 - 1);
                c[q] = mpo[f];
                at[q] = dst[f];
                z[q] = in[src[f]];
              }
#pragma unroll
              for (int q = 0; q < 4; ++q)
                if (e + q < e1) {
                  yr = fma(c[q].x, z[q].x, fma(-c[q].y, z[q].y, yr));
                  yi = fma(c[q].x, z[q].y, fma(c[q].y, z[q].x, yi));
                  if (at[q] >= 0) {
                    to[at[q]] = make_double2(yr, yi);
                    yr = yi = 0.0;
                  }
                }
            }
          }
        }
        lds_barrier();
        small_product<false>(g.g3, L, (const double2*)t2, same, out_at);
      } else {
        small_product<false>(g.g3, L, (const double2*)t1, same, out_at);
      }
      lds_barrier();
      // alpha_j, the update of w, beta_j with the breakdown test, v_{j+1} (k_lz_step), by the
      // waves that hold elements: the others would only take issue slots from them
      s = 0;
      if (mine) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const int i = t + e * NT;
          x[e] = make_double2(0.0, 0.0);
          if (i < n) {
            x[e] = wv[i];
            for (int p = 1; p < g.g3.ks; ++p) {
              const double2 z = wv[p * n + i];
              x[e].x += z.x;
              x[e].y += z.y;
            }
          }
          s += x[e].x * vc[e].x + x[e].y * vc[e].y;
        }
      }
      const double a = wg_sum(s, red[1], waves);
      const bool last = j + 1 == g.numiter, nfa = !isfinite(a);
      if (t == 0) {
        al[j] = a;
        if (nfa) { st[0] = last ? g.numiter : j + 1; st[2] = 1; }
      }
      if (last) break;
      s = 0;
      if (mine) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          x[e].x -= a * vc[e].x + b0 * vp[e].x;
          x[e].y -= a * vc[e].y + b0 * vp[e].y;
          s += x[e].x * x[e].x + x[e].y * x[e].y;
        }
      }
      s = wg_sum(s, red[2], waves);
      if (mine && !nfa) {
        const bool mid = s > 1e-280 && s < 1e280;
        const double inv = mid ? rsq_full(s) : 1.0 / sqrt(s), bn = mid ? s * inv : sqrt(s);
        const bool nfb = !isfinite(bn), brk = !nfb && bn < g.thresh;
        if (t == 0) {
          if (nfb) { st[0] = j + 1; st[2] = 1; }
          else if (brk) st[0] = st[1] = j + 1;
          else be[j] = bn;
        }
        if (!nfb && !brk) {
          b0 = bn;
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const int i = t + e * NT;
            vp[e] = vc[e];
            vc[e] = make_double2(div_by(x[e].x, bn, inv), div_by(x[e].y, bn, inv));
            if (i < n) v[i] = V[(int64_t)(j + 1) * g.js + i] = vc[e];
          }
        }
      }
      lds_barrier();
      if (st[1] | st[2]) break;
    }
  }
  __syncthreads();
  const int nvalid = st[0], nv = st[2] ? 0 : nvalid;
  if (t < 64) {
    double cr = 0.0, ci = 0.0, en = 0.0;
    bool conv = true;
    if (nv > 0)
      conv = tridiag_coefs(nv, al, be, (double*)t1, g.numiter | 1, g.mode, nrm, g.dt_re, g.dt_im,
                           cr, ci, en);
    if (t < nv) { cre[t] = cr; cim[t] = ci; }
    if (t == 0) { conv_s = conv; en_s = en; }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = t + e * NT;
    if (i < n) {
      double sr = 0.0, si = 0.0;
#pragma unroll 4
      for (int j = 0; j < nv; ++j) {
        const double2 z = V[(int64_t)j * g.js + i];
        sr += cre[j] * z.x - cim[j] * z.y;
        si += cre[j] * z.y + cim[j] * z.x;
      }
      g.out[(int64_t)b * n + i] = make_double2(sr, si);
    }
  }
  if (t == 0) {
    if (g.info) {
      int32_t* o = g.info + 4 * b;
      o[0] = nvalid;
      o[1] = st[1];
      o[2] = st[2] | (conv_s ? 0 : 2);
      o[3] = st[3];
    }
    if (g.energy) g.energy[b] = en_s;
  }
  if (g.alpha_beta && t < g.numiter) {
    double* ab = g.alpha_beta + (int64_t)2 * g.numiter * b;
    ab[t] = al[t];
    ab[g.numiter + t] = be[t];
  }
}

// Whether a solve fits the one-launch form, and its layout: FP64 without block
// structure (labels and masks keep their own products), T1, T2 and the vectors within LDS,
// a matvec of at most SMALL_FLOP.
static bool small_plan(const ptn_local_op* op, int numiter, int64_t batch, LzSmall* g) {
  if (op->precision != PTN_FP64) return false;
  const bool heff = op->kind == PTN_OP_HEFF;
  const int64_t d = heff ? op->d : 1;
  const int64_t top = 4096;
  if (op->Dl > top || op->Dr > top || d > top || op->Ml > top || op->Mr > top) return false;
  const int64_t n = op->Dl * d * op->Dr, n1 = op->Mr * op->Dr, n2 = d * op->Dr;
  if (n > SMALL_N) return false;
  const double flop = 8.0 * ((double)(op->Dl * d) * (double)n1 * (double)op->Dr +
                             (double)op->Dl * (double)n2 * (double)(op->Dl * op->Ml));
  if (flop * (double)((batch + SMALL_CUS - 1) / SMALL_CUS) > SMALL_FLOP || batch > 2 * SMALL_CUS)
    return false;
  const int64_t ni = d * op->Mr, no = op->Ml * d;
  if (heff && (ni > SMALL_MIX || no > SMALL_MIX)) return false;
  // 16 complex are all banks: rows of a multiple of 16 start half a turn apart
  auto pad = [](int64_t x) { return x % 16 ? x : x + 8; };
  g->heff = heff;
  g->Dl = (int)op->Dl;
  g->d = (int)d;
  g->Dr = (int)op->Dr;
  g->Ml = (int)op->Ml;
  g->Mr = (int)op->Mr;
  g->n = (int)n;
  g->numiter = numiter;
  g->ld1 = (int)(heff ? pad(n1) : n1);
  g->ld2 = (int)pad(n2);
  const int64_t z = ((int64_t)numiter * (numiter | 1) + 1) / 2;   // eigenvector matrix, over T1
  const int64_t s1 = op->Dl * d * g->ld1, s2 = heff ? op->Dl * op->Ml * g->ld2 : 4 * n;
  // the output product in parts of k while half of the waves would be idle; its
  // parts lie over T1 (H_eff) or behind it (bond)
  const int64_t tiles = (op->Dl + 15) / 16 * ((n2 + 7) / 8), steps = (op->Dl * op->Ml + 3) / 4;
  int ks = 1;
  while (ks < 4 && tiles * ks * 2 <= SHORT_T / 64 && steps >= 4 * ks && (!heff || 2 * ks * n <= s1)) ks *= 2;
  g->g1 = small_product_of(op->Dl * d, n1, op->Dr, op->Dr, 1, n1, 1);
  g->g3 = small_product_of(op->Dl, n2, op->Dl * op->Ml, 1, op->Dl, heff ? g->ld2 : n2, ks);
  g->rdr = 1.0f / (float)op->Dr;
  const int64_t up = (op->Dl * op->Dr + 63) / 64 * 64;
  g->parts = (int)std::max<int64_t>(1, std::min<int64_t>(SHORT_T / up, no));
  g->o_t1 = (int)n;
  g->o_t2 = (int)(n + std::max(s1, z));
  g->o_w = heff ? g->o_t1 : g->o_t2;
  g->o_mpo = (int)(g->o_t2 + s2);
  g->lds = 16 * (int)(g->o_mpo + (heff ? ni * no : 0));
  return g->lds <= SMALL_LDS;
}

static void small_solve(const LzSmall& g, int64_t batch, hipStream_t s) {
  const double flop = (double)batch * g.numiter * 8.0 * g.n *
                      ((double)g.Mr * g.Dr + (double)g.Dl * g.Ml);
  const dim3 B((unsigned)batch);
  tlaunch("k_lz_solve", flop, 0.0, k_lz_solve, B, dim3(SHORT_T), s, g);
}

}  // namespace ptn
