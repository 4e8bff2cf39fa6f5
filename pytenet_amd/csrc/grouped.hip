// Sector-grouped H_eff for U(1)-symmetric tensors: the two products of
// H_eff computed over the admissible quantum-number blocks only, each as ONE
// launch over all of its blocks.
//
// The tensors keep the reference's dense layout with zero blocks
// (pytenet/mps.py:71, pytenet/block_sparse_util.py:56-64). With quantum
// numbers ql (left virtual bond), qs (physical), qr (right virtual bond), qml /
// qmr (MPO virtual bonds) and the sign conventions of the reference's
// sparsity checks (pytenet/mps.py:71, pytenet/mpo.py:71,154,
// pytenet/tdvp.py:62) the nonzero entries are
//   A[l, s, r]          ql[l] + qs[s] = qr[r]
//   W[m, s', s, m']     qml[m] + qs[s'] = qs[s] + qmr[m']
//   R[r, m', r']        qr[r] + qmr[m'] = qr[r']
//   L[l, m, lb]         ql[l] + qml[m] = ql[lb]
// so that
//   T1[(l, s), (m', r')] = sum_r A[l, s, r] R[r, m', r'] is nonzero only where
//     ql[l] + qs[s] + qmr[m'] = qr[r'], and for fixed (s, m') and right
//     sector Q of r it is the dense block product
//       rows l in sector Q - qs[s], k = r in sector Q, columns r' in sector Q + qmr[m'];
//   out[lb, (s', r')] = sum_{(l, m)} L[l, m, lb] T2[(l, m), (s', r')] is nonzero only where
//     ql[lb] + qs[s'] = qr[r'], and for left sector P of lb and fixed s' it is
//       rows lb in P, columns r' in sector P + qs[s'], k over the segments
//       (l in sector P - qml[m], m), one segment per MPO index m.
// Every output block belongs to exactly one product block (its sector fixes
// the k-range), so no two workgroups write the same entry and no block needs
// accumulation. The entries of the output outside the blocks are structurally
// zero and are written by one fill pass; the sums inside a block run over
// exactly the reference's nonzero terms. The MPO mode mix between the products
// (k_mix_sectors) reads only the T1 entries the first product writes and writes
// only the T2 entries the second product reads.
//
// Launch: the grid covers the tiles of all blocks; a workgroup finds its block
// by binary search over the blocks' first tiles (descriptors in device memory,
// built once per distinct set of quantum numbers and kept in a cache).
// Requires the two virtual bonds to be sector-contiguous (each label in one
// run of indices), which the reference's QR and SVD splits produce
// (pytenet/block_sparse_util.py:106-180, 244-319); otherwise the tile-mask
// products are used.
#include <algorithm>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <unordered_map>
#include <utility>
#include <vector>
#include "gemm_impl.h"
#include "ops.h"

namespace ptn {

constexpr int GMAXSEG = 16;   // k-segments per block (MPO bond dimension at most 16)

struct GBlock {
  int64_t M, N;                 // block rows / columns (complex elements)
  int64_t c_off;                // element offset of the block in C
  int64_t tile0;                // first linear tile of the block in the launch
  int32_t tiles_n, nseg;
  int64_t a_off[GMAXSEG], b_off[GMAXSEG], K[GMAXSEG];
};

struct GLaunch {
  const GBlock* blocks;
  int nblocks;
  int64_t a_m, a_k, b_k, b_n, c_m, c_n;   // strides shared by all blocks
  const void* A;
  const void* B;
  void* C;
  const int* skip;
  int conjB;                              // B read conjugated
  // zero fill of the final output by fill_groups groups of FILL_GROUP workgroups spread over
  // this launch (the first product is bound by its matrix instructions, the fill by memory)
  double2* fill = nullptr;
  int64_t nfill = 0;
  unsigned fill_groups = 0;
  int64_t tiles = 0;                      // workgroups with a tile, when there is a fill
  int fast = 0;                           // byte offsets inside a tile's operands fit 32 bits
};
constexpr int64_t FILL_PER_WG = 16384;    // elements per fill workgroup
// Consecutive workgroups go to the 8 XCDs and their 4 shader engines each in turn. Fill
// workgroups at single even distances can fall on the same engines for long stretches, which
// leaves the tiles to the others (1280 among 1452 tiles: some engines get 1.9 times their share
// of 768 in a row); groups of 32 take one place of each. Left environment step at D = 2048 with
// three sectors of 683, FP64: first product 2119 -> 1185 us (1174 and a fill launch of 55), the
// step 3550 -> 2590 us, in FP32 2090 -> 1560 us.
constexpr unsigned FILL_GROUP = 32;

// One workgroup = one BM x BN tile of one block; staging and MFMA steps are those of
// zgemm_kernel (whole complex elements, uniform bases with constant 32-bit
// offsets, rows and columns beyond the block clamped to its last ones, only the
// partial last stage of a segment with predicates), with k running over the block's
// segments. Two-site H_eff at D = 2048 (U(1)): first product 249 -> 232 us, output product
// 305 -> 232 us.
template <typename Tc, typename TA, typename TB, typename TC, int TM, int TN, bool A_KCONTIG,
          bool B_NCONTIG>
__global__ __launch_bounds__(256) void zgemm_grouped_kernel(GLaunch g) {
  typedef TileCfg<TM, TN, StageK<Tc, TM>::value> T;
  constexpr int BM = T::BM, BN = T::BN, BK = T::BK, NA = T::NA, NB = T::NB;
  typedef typename acc4<Tc>::type acc_t;
  typedef typename cplx_of<Tc>::type C2;
  __shared__ __align__(16) C2 As[2][BK][BM + 1];
  __shared__ __align__(16) C2 Bs[2][BK][BN + 1];
  if (g.skip && g.skip[0]) return;
  // the fill's groups come at even distances among the tiles' ones
  int64_t tile = blockIdx.x;
  if (g.fill_groups) {
    const uint64_t grp = blockIdx.x / FILL_GROUP, all = gridDim.x / FILL_GROUP;
    const uint64_t f = grp * g.fill_groups / all;
    if ((grp + 1) * g.fill_groups / all > f) {
      const int64_t i0 = (int64_t)(f * FILL_GROUP + blockIdx.x % FILL_GROUP) * FILL_PER_WG;
      const int64_t e = i0 + FILL_PER_WG < g.nfill ? i0 + FILL_PER_WG : g.nfill;
      for (int64_t i = i0 + threadIdx.x; i < e; i += 256) g.fill[i] = make_double2(0.0, 0.0);
      return;
    }
    tile -= (int64_t)f * FILL_GROUP;
    if (tile >= g.tiles) return;
  }
  // the block of this workgroup: the last block whose first tile <= its tile
  int lo = 0, hi = g.nblocks - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (g.blocks[mid].tile0 <= tile) lo = mid; else hi = mid - 1;
  }
  const GBlock* __restrict__ bk = g.blocks + lo;
  const int64_t bM = bk->M, bN = bk->N;
  const int nseg = bk->nseg;
  const int64_t lt = tile - bk->tile0;
  const int64_t m0 = (lt / bk->tiles_n) * BM, n0 = (lt % bk->tiles_n) * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm0 = (wave >> 1) * T::WM, wn0 = (wave & 1) * T::WN;
  const TA* __restrict__ A = (const TA*)g.A + m0 * g.a_m;
  const TB* __restrict__ B = (const TB*)g.B + n0 * g.b_n;
  TC* __restrict__ C = (TC*)g.C + bk->c_off;
  const Tc sb = g.conjB ? (Tc)-1 : (Tc)1;

  auto arow = [&](int i) -> int { return A_KCONTIG ? (tid + 256 * i) / BK : (tid + 256 * i) % BM; };
  auto ak = [&](int i) -> int { return A_KCONTIG ? (tid + 256 * i) % BK : (tid + 256 * i) / BM; };
  auto bcol = [&](int i) -> int { return B_NCONTIG ? (tid + 256 * i) % BN : (tid + 256 * i) / BK; };
  auto bkk = [&](int i) -> int { return B_NCONTIG ? (tid + 256 * i) / BN : (tid + 256 * i) % BK; };
  const int mlast = (int)(bM - m0 < BM ? bM - m0 : BM) - 1;
  const int nlast = (int)(bN - n0 < BN ? bN - n0 : BN) - 1;
  uint32_t offa[NA], offb[NB];
#pragma unroll
  for (int i = 0; i < NA; ++i)
    offa[i] = (uint32_t)((min(arow(i), mlast) * g.a_m + ak(i) * g.a_k) * (int64_t)sizeof(TA));
#pragma unroll
  for (int i = 0; i < NB; ++i)
    offb[i] = (uint32_t)((min(bcol(i), nlast) * g.b_n + bkk(i) * g.b_k) * (int64_t)sizeof(TB));

  // the next stage to load: segment sg, k offset k0 in it
  int sg = 0;
  int64_t k0 = 0, K = bk->K[0];
  const TA* Ap = A + bk->a_off[0];
  const TB* Bp = B + bk->b_off[0];
  int nst = 0;
  for (int i = 0; i < nseg; ++i) nst += (int)((bk->K[i] + BK - 1) / BK);
  C2 ra[NA], rb[NB];
  auto load_next = [&]() {
    const TA* Ak = Ap + k0 * g.a_k;
    const TB* Bk = Bp + k0 * g.b_k;
    if (g.fast && k0 + BK <= K) {
#pragma unroll
      for (int i = 0; i < NA; ++i)
        load_c<Tc>((const TA*)((const char*)Ak + offa[i]), ra[i].x, ra[i].y);
#pragma unroll
      for (int i = 0; i < NB; ++i)
        load_c<Tc>((const TB*)((const char*)Bk + offb[i]), rb[i].x, rb[i].y);
    } else {
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        ra[i] = C2{0, 0};
        if (k0 + ak(i) < K)
          load_c<Tc>(Ak + (int64_t)min(arow(i), mlast) * g.a_m + (int64_t)ak(i) * g.a_k, ra[i].x,
                     ra[i].y);
      }
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        rb[i] = C2{0, 0};
        if (k0 + bkk(i) < K)
          load_c<Tc>(Bk + (int64_t)min(bcol(i), nlast) * g.b_n + (int64_t)bkk(i) * g.b_k, rb[i].x,
                     rb[i].y);
      }
    }
    k0 += BK;
    if (k0 >= K && sg + 1 < nseg) {
      ++sg;
      k0 = 0;
      K = bk->K[sg];
      Ap = A + bk->a_off[sg];
      Bp = B + bk->b_off[sg];
    }
  };
  auto store_tiles = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NA; ++i) As[buf][ak(i)][arow(i)] = ra[i];
#pragma unroll
    for (int i = 0; i < NB; ++i) Bs[buf][bkk(i)][bcol(i)] = C2{rb[i].x, sb * rb[i].y};
  };

  acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
  const int l16 = lane & 15, kk = lane >> 4, pb = lane & 1;
  int buf = 0;
  if (nst > 0) {
    load_next();
    store_tiles(0);
  }
  __syncthreads();
  for (int it = 0; it < nst; ++it) {
    const bool more = it + 1 < nst;
    if (more) load_next();
#pragma unroll
    for (int ks = 0; ks < BK / 4; ++ks) {
      C2 av[TM];
      Tc b0[TN], b1[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) av[i] = As[buf][4 * ks + kk][wm0 + 16 * i + l16];
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const C2 b = Bs[buf][4 * ks + kk][wn0 + 8 * j + (l16 >> 1)];
        b0[j] = pb ? b.y : b.x;
        b1[j] = pb ? b.x : -b.y;
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mfma16(av[i].x, b0[j], acc[i][j]);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mfma16(av[i].y, b1[j], acc[i][j]);
    }
    if (more) store_tiles(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
  // epilogue as zgemm_kernel: the partner lane (lane ^ 1) holds the other part
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      Tc mine[4], other[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        mine[v] = acc[i][j][v];
        other[v] = __shfl_xor(mine[v], 1);
      }
      const int64_t n = n0 + wn0 + 8 * j + ((lane & 15) >> 1);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int v = 2 * pb + h;
        const int64_t m = m0 + wm0 + 16 * i + acc4<Tc>::row(kk, v);
        const double re = pb ? (double)other[2 + h] : (double)mine[h];
        const double im = pb ? (double)mine[2 + h] : (double)other[h];
        if (m < bM && n < bN) store_c(C + m * g.c_m + n * g.c_n, re, im);
      }
    }
  }
}

// zero fill of n complex elements (the structurally zero entries of the output)
template <typename TC>
__global__ void k_zero_fill(int64_t n, TC* __restrict__ p, const int* __restrict__ skip) {
  if (skip && skip[0]) return;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
       t += (int64_t)gridDim.x * blockDim.x)
    store_c(p + t, 0.0, 0.0);
}

template <typename TC>
static int zero_fill(int64_t n, void* p, hipStream_t s) {
  if (n <= 0) return PTN_OK;
  int64_t b = (n + 255) / 256;
  if (b > 4096) b = 4096;
  tlaunch("k_zero_fill", 0.0, (double)n * sizeof(TC), k_zero_fill<TC>, dim3((unsigned)b),
          dim3(256), s, n, (TC*)p, skip_flag().p);
  PTN_LAUNCH_CHECK();
  return PTN_OK;
}

// ---------------------------------------------------------------------------
// Sector-aware MPO mode mix T2[l, o, r'] = sum_i Wm[o, i] T1[l, i, r'] with
// i = (s, m'), o = (m, s'). For a left sector P of l and a right sector Q of
// r' (a "unit"), T1[l, i, r'] is nonzero only for the inputs i with
// qs[s] + qmr[m'] = Q - P whose k-sector P + qs[s] exists (exactly the entries
// the first grouped product writes), and the second product reads T2[l, o, r']
// only for the outputs o with qml[m] + qs[s'] = Q - P whose output sector
// P + qml[m] exists. The mix reads and writes just those: T1 needs no zero
// fill and T2 no zeros outside what is read. A workgroup takes MIX_ROWS rows l of one
// 64-column chunk of a unit, MIX_ROWS / 4 per wave, the lanes over the columns r'
// (coalesced). Memory-bound, so what counts is the bytes in flight per CU and
// little else per byte: the unit's part of W is gathered once per workgroup, a lane's
// inputs are held in registers sized to the plan's longest input list (CAP = 8, 16 or
// 32), the next row's loaded while the current one is mixed, and complex64
// operands are mixed in FP32 arithmetic (A = float). D = 2048: 72 -> 58 us.
constexpr int MIX_LIST = 32;   // d * Mr and Ml * d are at most 32
enum { PLAN_HEFF = SECTORS_HEFF, PLAN_ENV_RIGHT = SECTORS_ENV_RIGHT, PLAN_ENV_LEFT = SECTORS_ENV_LEFT };

struct MixUnit {
  int64_t l0, nl, r0, nr;
  int64_t tile0;                // first workgroup of the unit
  int32_t ni, no;
  int32_t chunks;               // 64-column chunks per row
  int8_t il[MIX_LIST], ol[MIX_LIST];
};
constexpr int MIX_ROWS = 16;    // rows per workgroup

template <typename TX, typename TY, typename A, int CAP>
__global__ __launch_bounds__(256) void k_mix_sectors(const MixUnit* __restrict__ units, int nunits,
                                                     int ni_all, int no_all, int64_t nr_all,
                                                     const double2* __restrict__ wm,
                                                     const TX* __restrict__ x, TY* __restrict__ y,
                                                     const int* __restrict__ skip, int wtrans) {
  typedef typename cplx_of<A>::type C2;
  __shared__ C2 W[MIX_LIST * MIX_LIST];
  __shared__ int il[MIX_LIST], ol[MIX_LIST];
  if (skip && skip[0]) return;
  const int64_t tile = blockIdx.x;
  int lo = 0, hi = nunits - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (units[mid].tile0 <= tile) lo = mid; else hi = mid - 1;
  }
  const MixUnit* __restrict__ u = units + lo;
  const int ni = u->ni, no = u->no;
  if (threadIdx.x < MIX_LIST) il[threadIdx.x] = u->il[threadIdx.x];
  else if (threadIdx.x < 2 * MIX_LIST) ol[threadIdx.x - MIX_LIST] = u->ol[threadIdx.x - MIX_LIST];
  __syncthreads();
  // Wm[o, i] of the unit's lists, or stored transposed as W[i, o] (left environment)
  for (int t = threadIdx.x; t < ni * no; t += 256) {
    const int j = t / ni, k = t - j * ni;
    const int o = ol[j], i = il[k];
    const double2 w = wtrans ? wm[i * no_all + o] : wm[o * ni_all + i];
    W[t] = C2{(A)w.x, (A)w.y};
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t rt = tile - u->tile0;
  const int64_t row0 = rt / u->chunks * MIX_ROWS;
  const int64_t c = rt % u->chunks * 64 + lane;
  const bool in = c < u->nr;
  const int64_t r = u->r0 + c;
  const int64_t rows = u->nl - row0 < MIX_ROWS ? u->nl - row0 : MIX_ROWS;
  const int64_t l0 = u->l0 + row0;
  // the lanes share the lists: offsets in scalar registers, known before the loads
  int64_t ioff[CAP];
#pragma unroll
  for (int k = 0; k < CAP; ++k)
    ioff[k] = (int64_t)__builtin_amdgcn_readfirstlane(k < ni ? il[k] : 0) * nr_all;
  C2 next[CAP];
  auto load = [&](int64_t row) {
    const TX* __restrict__ xl = x + (l0 + row) * ni_all * nr_all + r;
#pragma unroll
    for (int k = 0; k < CAP; ++k) {
      next[k] = C2{0, 0};
      if (k < ni && in) load_c<A>(xl + ioff[k], next[k].x, next[k].y);
    }
  };
  if (wave < rows) load(wave);
  for (int64_t row = wave; row < rows; row += 4) {
    C2 v[CAP];
#pragma unroll
    for (int k = 0; k < CAP; ++k) v[k] = next[k];
    if (row + 4 < rows) load(row + 4);
    TY* __restrict__ yl = y + (l0 + row) * no_all * nr_all + r;
    for (int j = 0; j < no; ++j) {
      A yr = 0, yi = 0;
#pragma unroll
      for (int k = 0; k < CAP; ++k) {
        if (k < ni) {
          const C2 w = W[j * ni + k];
          yr += w.x * v[k].x - w.y * v[k].y;
          yi += w.x * v[k].y + w.y * v[k].x;
        }
      }
      if (in) store_c(yl + (int64_t)ol[j] * nr_all, yr, yi);
    }
  }
}

// ---------------------------------------------------------------------------
// plans: the blocks of both products for one set of quantum numbers

struct Sector { int64_t start, len; };

// runs of equal labels of a bond; false if a label has two runs
static bool sectors_of(const int64_t* q, int64_t n, std::map<int64_t, Sector>& out) {
  out.clear();
  for (int64_t i = 0; i < n;) {
    int64_t j = i;
    while (j < n && q[j] == q[i]) ++j;
    if (out.count(q[i])) return false;
    out[q[i]] = Sector{i, j - i};
    i = j;
  }
  return true;
}

struct GProduct {
  std::vector<GBlock> blocks;
  std::vector<std::pair<int64_t, int32_t>> order;   // (-K, block), as uploaded
  int64_t tiles = 0;
  int tile = 2;         // TileCfg<tile, tile>: 128 x 64 (4), 64 x 32 (2) or 32 x 16 (1)
  double flop = 0.0;    // 8 M N K summed over the blocks
  double bytes = 0.0;   // operand blocks read once, output blocks written once
};

struct SectorPlan {
  SectorPlan() = default;
  SectorPlan(const SectorPlan&) = delete;
  SectorPlan& operator=(const SectorPlan&) = delete;
  // the descriptors are freed with the plan's last reference (hipFree waits
  // for the device, so no launch still reads them)
  ~SectorPlan() {
    if (dev) {
      int cur = 0;
      if (hipGetDevice(&cur) == hipSuccess && cur != device) (void)hipSetDevice(device);
      (void)hipFree(dev);
      if (cur != device) (void)hipSetDevice(cur);
    }
  }
  int kind = PLAN_HEFF;
  GProduct p1, p3;
  std::vector<MixUnit> mix;
  int64_t mix_tiles = 0;
  double mix_bytes = 0.0;   // T1 entries read and T2 entries written by the mix (elements)
  int mix_cap = MIX_LIST;   // register capacity for a unit's inputs (8, 16 or 32)
  GBlock* dev = nullptr;    // p1's blocks, then p3's, then the mix units
  MixUnit* dev_mix = nullptr;
  int device = 0;
  uint64_t stamp = 0;
};

// Tile shape and first tiles of a product. The 128 x 64 tile when its padding
// costs at most 15 % more work than the 64 x 32 tile's and it still gives
// enough workgroups for the chip (>= 512); else the cheaper of 64 x 32 and 32 x 16 by
// padded work / (rate x share of the chip at work): full tiles of them reach 63 and
// 52 TFLOP/s (FP64), and with fewer than about six tiles per CU the CUs that get
// one more than the others set the time. Two-site U(1) H_eff, both products on 64 x 32
// against both on 32 x 16 tiles: D = 96 40 / 35 us, 512 78 / 59, 1024 138 / 112,
// 1500 261 / 248, 2048 493 / 503 (and 473 with the output product alone on 32 x 16:
// 811 tiles of 64 x 32 are 3.2 per CU).
// FP32 products take the choice of the FP64 rates, which was not measured tile by
// tile there: with the staging of this kernel two-site H_eff in FP32 went from 41 to 38 us at D = 96, 100 to 68
// at 512, 219 to 167 at 1024 and 784 to 668 at 2048.
static void finish_product(GProduct& P, size_t csz_a, size_t csz_b, size_t csz_c) {
  static const struct { int code; int64_t bm, bn; double rate; } tile[3] = {
      {4, 128, 64, 65.0}, {2, 64, 32, 63.0}, {1, 32, 16, 52.0}};
  double work[3] = {0, 0, 0};
  int64_t n[3] = {0, 0, 0};
  P.flop = 0.0;
  P.bytes = 0.0;
  auto up = [](int64_t x, int64_t t) { return (x + t - 1) / t * t; };
  auto total_k = [](const GBlock& b) {
    int64_t k = 0;
    for (int i = 0; i < b.nseg; ++i) k += b.K[i];
    return k;
  };
  for (const GBlock& b : P.blocks) {
    const double k = (double)total_k(b);
    P.flop += 8.0 * (double)b.M * (double)b.N * k;
    P.bytes += k * ((double)b.M * csz_a + (double)b.N * csz_b) + (double)b.M * b.N * csz_c;
    for (int t = 0; t < 3; ++t) {
      const int64_t m = up(b.M, tile[t].bm), c = up(b.N, tile[t].bn);
      work[t] += (double)m * (double)c * k;
      n[t] += (m / tile[t].bm) * (c / tile[t].bn);
    }
  }
  int pick = 0;
  if (!(work[0] <= 1.15 * work[1] && n[0] >= 512)) {
    auto cost = [&](int t) {
      return n[t] ? work[t] / tile[t].rate * (double)up(n[t], 256) / (double)n[t] : 0.0;
    };
    pick = cost(2) < cost(1) ? 2 : 1;
  }
  P.tile = tile[pick].code;
  // the tiles with the longest sums first, so that the last workgroups are short ones: the
  // blocks' order in the device array (the descriptors themselves are 424 bytes each)
  P.order.resize(P.blocks.size());
  for (size_t i = 0; i < P.blocks.size(); ++i) P.order[i] = {-total_k(P.blocks[i]), (int32_t)i};
  std::sort(P.order.begin(), P.order.end());
  int64_t tiles = 0;
  for (const auto& o : P.order) {
    GBlock& b = P.blocks[o.second];
    b.tiles_n = (int32_t)((b.N + tile[pick].bn - 1) / tile[pick].bn);
    b.tile0 = tiles;
    tiles += ((b.M + tile[pick].bm - 1) / tile[pick].bm) * b.tiles_n;
  }
  P.tiles = tiles;
}

using SectorMap = std::map<int64_t, Sector>;

static GBlock block(int64_t M, int64_t N, int64_t c_off) {
  GBlock b{};
  b.M = M;
  b.N = N;
  b.c_off = c_off;
  return b;
}
static void add_segment(GBlock& b, int64_t a_off, int64_t b_off, int64_t K) {
  b.a_off[b.nseg] = a_off;
  b.b_off[b.nseg] = b_off;
  b.K[b.nseg] = K;
  ++b.nseg;
}

// T1[(l, s), (m', r')] = sum_r A[(l, s), r] R[r, (m', r')] (H_eff and the
// right environment step): block per (s, right sector Q of r, m')
static void plan_a_times_r(const Dims& D, const int64_t* qs, const int64_t* qmr,
                           const SectorMap& sl, const SectorMap& sr, GProduct& P) {
  for (int64_t s = 0; s < D.d; ++s)
    for (const auto& kq : sr) {
      const auto itl = sl.find(kq.first - qs[s]);
      if (itl == sl.end()) continue;
      for (int64_t mp = 0; mp < D.Mr; ++mp) {
        const auto itc = sr.find(kq.first + qmr[mp]);
        if (itc == sr.end()) continue;
        const int64_t l0 = itl->second.start, r0 = kq.second.start, c0 = itc->second.start;
        GBlock b = block(itl->second.len, itc->second.len,
                         (l0 * D.d + s) * (D.Mr * D.Dr) + mp * D.Dr + c0);
        add_segment(b, (l0 * D.d + s) * D.Dr + r0, r0 * (D.Mr * D.Dr) + mp * D.Dr + c0,
                    kq.second.len);
        P.blocks.push_back(b);
      }
    }
}

// H_eff: out[lb, (s', r')] = sum_{(l, m)} L[(l, m), lb] T2[(l, m), (s', r')]:
// block per (left sector P of lb, s'), one k-segment per MPO index m
static void plan_heff_out(const Dims& D, const int64_t* qs, const int64_t* qml,
                          const SectorMap& sl, const SectorMap& sr, GProduct& P) {
  for (const auto& pq : sl) {
    const int64_t lb0 = pq.second.start;
    for (int64_t s2 = 0; s2 < D.d; ++s2) {
      const auto itc = sr.find(pq.first + qs[s2]);
      if (itc == sr.end()) continue;
      const int64_t c0 = itc->second.start;
      GBlock b = block(pq.second.len, itc->second.len, lb0 * (D.d * D.Dr) + s2 * D.Dr + c0);
      for (int64_t m = 0; m < D.Ml; ++m) {
        const auto itl = sl.find(pq.first - qml[m]);
        if (itl == sl.end()) continue;
        const int64_t l0 = itl->second.start;
        add_segment(b, (l0 * D.Ml + m) * D.Dl + lb0, (l0 * D.Ml + m) * (D.d * D.Dr) + s2 * D.Dr + c0,
                    itl->second.len);
      }
      if (b.nseg) P.blocks.push_back(b);   // no segment: a structurally zero block
    }
  }
}

// right environment: out[(l, m), lb] = sum_{(s', r')} T2[(l, m), (s', r')] conj(B[lb, (s', r')]):
// block per (left sector P of l, m), one k-segment per physical index s'
static void plan_envr_out(const Dims& D, const int64_t* qs, const int64_t* qml,
                          const SectorMap& sl, const SectorMap& sr, GProduct& P) {
  for (const auto& pq : sl) {
    const int64_t l0 = pq.second.start;
    for (int64_t m = 0; m < D.Ml; ++m) {
      const auto itb = sl.find(pq.first + qml[m]);
      if (itb == sl.end()) continue;
      const int64_t lb0 = itb->second.start;
      GBlock b = block(pq.second.len, itb->second.len, (l0 * D.Ml + m) * D.Dl + lb0);
      for (int64_t s2 = 0; s2 < D.d; ++s2) {
        const auto itr = sr.find(itb->first + qs[s2]);
        if (itr == sr.end()) continue;
        const int64_t rb0 = itr->second.start;
        add_segment(b, (l0 * D.Ml + m) * (D.d * D.Dr) + s2 * D.Dr + rb0,
                    lb0 * (D.d * D.Dr) + s2 * D.Dr + rb0, itr->second.len);
      }
      if (b.nseg) P.blocks.push_back(b);
    }
  }
}

// left environment: T1[(l, m), (s', r')] = sum_lb L[(l, m), lb] conj(B[lb, (s', r')]):
// block per (left sector P of l, m, s')
static void plan_l_times_b(const Dims& D, const int64_t* qs, const int64_t* qml,
                           const SectorMap& sl, const SectorMap& sr, GProduct& P) {
  for (const auto& pq : sl) {
    const int64_t l0 = pq.second.start;
    for (int64_t m = 0; m < D.Ml; ++m) {
      const auto itb = sl.find(pq.first + qml[m]);
      if (itb == sl.end()) continue;
      const int64_t lb0 = itb->second.start;
      for (int64_t s2 = 0; s2 < D.d; ++s2) {
        const auto itr = sr.find(itb->first + qs[s2]);
        if (itr == sr.end()) continue;
        const int64_t rb0 = itr->second.start;
        GBlock b = block(pq.second.len, itr->second.len,
                         (l0 * D.Ml + m) * (D.d * D.Dr) + s2 * D.Dr + rb0);
        add_segment(b, (l0 * D.Ml + m) * D.Dl + lb0, lb0 * (D.d * D.Dr) + s2 * D.Dr + rb0,
                    itb->second.len);
        P.blocks.push_back(b);
      }
    }
  }
}

// left environment: out[r, (m', r')] = sum_{(l, s)} A[(l, s), r] T2[(l, s), (m', r')]:
// block per (right sector Q of r, m'), one k-segment per physical index s
static void plan_envl_out(const Dims& D, const int64_t* qs, const int64_t* qmr,
                          const SectorMap& sl, const SectorMap& sr, GProduct& P) {
  for (const auto& rq : sr) {
    const int64_t r0 = rq.second.start;
    for (int64_t mp = 0; mp < D.Mr; ++mp) {
      const auto itc = sr.find(rq.first + qmr[mp]);
      if (itc == sr.end()) continue;
      const int64_t c0 = itc->second.start;
      GBlock b = block(rq.second.len, itc->second.len, r0 * (D.Mr * D.Dr) + mp * D.Dr + c0);
      for (int64_t s = 0; s < D.d; ++s) {
        const auto itl = sl.find(rq.first - qs[s]);
        if (itl == sl.end()) continue;
        const int64_t l0 = itl->second.start;
        add_segment(b, (l0 * D.d + s) * D.Dr + r0, (l0 * D.d + s) * (D.Mr * D.Dr) + mp * D.Dr + c0,
                    itl->second.len);
      }
      if (b.nseg) P.blocks.push_back(b);
    }
  }
}

// mix units for a unit (left sector P, right sector Q, dq = Q - P):
// H_eff / right environment: inputs i = (s, m') with qs[s] + qmr[m'] = dq and
// k-sector P + qs[s] present, outputs o = (m, s') with qml[m] + qs[s'] = dq and
// P + qml[m] present; left environment: inputs i = (m, s') with
// qml[m] + qs[s'] = dq and P + qml[m] present, outputs o = (s, m') with
// qs[s] + qmr[m'] = dq and P + qs[s] present.
static void plan_mix(const Dims& D, bool left, const int64_t* qs, const int64_t* qml,
                     const int64_t* qmr, const SectorMap& sl, const SectorMap& sr,
                     SectorPlan& sp) {
  for (const auto& pq : sl)
    for (const auto& rq : sr) {
      const int64_t P = pq.first, dq = rq.first - P;
      MixUnit u{};
      int8_t* sm_list = left ? u.il : u.ol;    // (m, s') indices
      int8_t* ms_list = left ? u.ol : u.il;    // (s, m') indices
      int32_t& n_sm = left ? u.ni : u.no;
      int32_t& n_ms = left ? u.no : u.ni;
      for (int64_t m = 0; m < D.Ml; ++m)
        for (int64_t s2 = 0; s2 < D.d; ++s2)
          if (qml[m] + qs[s2] == dq && sl.count(P + qml[m])) sm_list[n_sm++] = (int8_t)(m * D.d + s2);
      for (int64_t s1 = 0; s1 < D.d; ++s1)
        for (int64_t mp = 0; mp < D.Mr; ++mp)
          if (qs[s1] + qmr[mp] == dq && sr.count(P + qs[s1])) ms_list[n_ms++] = (int8_t)(s1 * D.Mr + mp);
      if (u.no == 0) continue;   // nothing of this unit is read
      u.l0 = pq.second.start;
      u.nl = pq.second.len;
      u.r0 = rq.second.start;
      u.nr = rq.second.len;
      u.tile0 = sp.mix_tiles;
      u.chunks = (int32_t)((u.nr + 63) / 64);
      sp.mix_tiles += (u.nl + MIX_ROWS - 1) / MIX_ROWS * u.chunks;
      sp.mix_bytes += (double)u.nl * (double)u.nr * (double)(u.ni + u.no);
      sp.mix.push_back(u);
    }
}

// blocks of both products and the mix units of a plan kind; false when a bond
// is not sector-contiguous, a segment or mix list would exceed its limit, or
// the launch would be too large
static bool build_plan(int kind, const Dims& D, const int64_t* ql, const int64_t* qs,
                       const int64_t* qr, const int64_t* qml, const int64_t* qmr, size_t csz,
                       SectorPlan& sp) {
  if (D.Dl <= 0 || D.Dr <= 0 || D.d <= 0 || D.Ml <= 0 || D.Mr <= 0 ||
      D.d * D.Mr > MIX_LIST || D.Ml * D.d > MIX_LIST)
    return false;
  if ((kind == PLAN_HEFF && D.Ml > GMAXSEG) || (kind != PLAN_HEFF && D.d > GMAXSEG)) return false;
  SectorMap sl, sr;
  if (!sectors_of(ql, D.Dl, sl) || !sectors_of(qr, D.Dr, sr)) return false;
  sp.kind = kind;
  if (kind == PLAN_ENV_LEFT) {
    plan_l_times_b(D, qs, qml, sl, sr, sp.p1);
    plan_mix(D, true, qs, qml, qmr, sl, sr, sp);
    plan_envl_out(D, qs, qmr, sl, sr, sp.p3);
    finish_product(sp.p1, csz, 16, csz);   // L in the compute type, B complex128
    finish_product(sp.p3, 16, csz, 16);    // A and out complex128
  } else {
    plan_a_times_r(D, qs, qmr, sl, sr, sp.p1);
    plan_mix(D, false, qs, qml, qmr, sl, sr, sp);
    if (kind == PLAN_HEFF) {
      plan_heff_out(D, qs, qml, sl, sr, sp.p3);
      finish_product(sp.p3, csz, csz, 16);
    } else {
      plan_envr_out(D, qs, qml, sl, sr, sp.p3);
      finish_product(sp.p3, csz, 16, 16);
    }
    finish_product(sp.p1, 16, csz, csz);   // A complex128, R and T1 in the compute type
  }
  int maxni = 0;
  for (const MixUnit& u : sp.mix) maxni = u.ni > maxni ? u.ni : maxni;
  sp.mix_cap = maxni <= 8 ? 8 : (maxni <= 16 ? 16 : MIX_LIST);
  return sp.p1.tiles > 0 && sp.p3.tiles > 0 && sp.p1.tiles < 0x7fffffff &&
         sp.p3.tiles < 0x7fffffff && !sp.mix.empty() && sp.mix_tiles < 0x7fffffff;
}

// arithmetic of the grouped products for a precision code: FP64 or FP32
// (the three-term split-bf16 mode has FP32 accuracy and takes the FP32
// products); -1 when they do not apply (two-term split-bf16: the tile-mask
// products)
static int grouped_prec(int prec) {
  const int bp = prec & ~PTN_BLOCK_SPARSE;
  if (bp == PTN_FP64) return PTN_FP64;
  if (bp == PTN_FP32 || bp == PTN_BF16X6) return PTN_FP32;
  return -1;
}

namespace {
std::mutex g_plan_mu;
// nullptr: not applicable. Allocated once and never destroyed, so that no
// plan is released (hipFree) during static destruction at process exit, when
// the HIP runtime may already be gone.
auto& g_plans = *new std::unordered_map<std::string, std::shared_ptr<SectorPlan>>();
uint64_t g_plan_clock = 0;
constexpr size_t PLAN_CACHE_MAX = 1024;
}  // namespace

static void append(std::string& k, const int64_t* p, int64_t n) {
  k.append((const char*)&n, sizeof(n));
  k.append((const char*)p, (size_t)n * sizeof(int64_t));
}

// The sector plan of kind PLAN_* for a site operator with quantum numbers
// (null when the operator has none, is not a site operator, or the grouped
// products do not apply). Builds and uploads it on first use (synchronous
// copy: call it outside stream capture); plans are cached per device, kind
// and set of quantum numbers.
int sector_plan_get(const ptn_local_op* op, int kind, SectorPlanRef* out) {
  out->reset();
  if (!op || op->kind != PTN_OP_HEFF || !(op->precision & PTN_BLOCK_SPARSE) || !op->q_l ||
      !op->q_s || !op->q_r || !op->q_ml || !op->q_mr)
    return PTN_OK;
  const int bp = grouped_prec(op->precision);
  if (bp < 0) return PTN_OK;
  if (noalloc_mode()) return PTN_OK;
  int dev = 0;
  PTN_HIP_CHECK(hipGetDevice(&dev));
  std::string key;
  const int64_t head[8] = {dev, bp, kind, op->Dl, op->d, op->Dr, op->Ml, op->Mr};
  key.append((const char*)head, sizeof(head));
  append(key, op->q_l, op->Dl);
  append(key, op->q_s, op->d);
  append(key, op->q_r, op->Dr);
  append(key, op->q_ml, op->Ml);
  append(key, op->q_mr, op->Mr);
  std::lock_guard<std::mutex> lk(g_plan_mu);
  auto it = g_plans.find(key);
  if (it != g_plans.end()) {
    if (it->second) it->second->stamp = ++g_plan_clock;
    *out = it->second;
    return PTN_OK;
  }
  if (g_plans.size() >= PLAN_CACHE_MAX) {
    // drop the older half of this device's plans from the cache (a plan still
    // held by a caller lives on until that caller releases it)
    std::vector<std::pair<uint64_t, std::string>> age;
    for (auto& kv : g_plans)
      if (!kv.second || kv.second->device == dev)
        age.emplace_back(kv.second ? kv.second->stamp : 0, kv.first);
    std::sort(age.begin(), age.end());
    for (size_t i = 0; i < age.size() / 2; ++i) g_plans.erase(age[i].second);
  }
  std::shared_ptr<SectorPlan> sp(new SectorPlan());
  const Dims D = {op->Dl, op->d, op->Dr, op->Ml, op->Mr};
  if (!build_plan(kind, D, op->q_l, op->q_s, op->q_r, op->q_ml, op->q_mr,
                  bp == PTN_FP64 ? 16 : 8, *sp)) {
    g_plans.emplace(key, nullptr);
    return PTN_OK;
  }
  std::vector<GBlock> all;
  all.reserve(sp->p1.blocks.size() + sp->p3.blocks.size());
  for (const GProduct* p : {&sp->p1, &sp->p3})
    for (const auto& o : p->order) all.push_back(p->blocks[o.second]);
  const size_t bb = (all.size() * sizeof(GBlock) + 255) & ~(size_t)255;
  const size_t mb = sp->mix.size() * sizeof(MixUnit);
  hipError_t e = hipMalloc((void**)&sp->dev, bb + mb);
  if (e == hipSuccess) e = hipMemcpy(sp->dev, all.data(), all.size() * sizeof(GBlock),
                                     hipMemcpyHostToDevice);
  sp->dev_mix = (MixUnit*)((char*)sp->dev + bb);
  if (e == hipSuccess) e = hipMemcpy(sp->dev_mix, sp->mix.data(), mb, hipMemcpyHostToDevice);
  sp->device = dev;
  if (e != hipSuccess) {
    ptn_set_last_hip_error(e);
    return PTN_ERR_HIP;   // the plan (and its allocation) is released here
  }
  sp->stamp = ++g_plan_clock;
  *out = sp;
  g_plans.emplace(key, std::move(sp));
  return PTN_OK;
}

template <typename Tc, typename TA, typename TB, typename TC, bool AK, bool BNC>
static int grouped_launch(GLaunch g, const GProduct& P, hipStream_t s) {
  // launch records keep the name pointer: formatted once per instance
  static const auto make = [](int t) {
    char name[112];
    snprintf(name, sizeof(name), "zgemm_grouped_kernel<%s, %s, %s, %s, %d, %d, %s, %s>",
             type_tag<Tc>::s, type_tag<TA>::s, type_tag<TB>::s, type_tag<TC>::s, t, t,
             AK ? "true" : "false", BNC ? "true" : "false");
    return std::string(name);
  };
  static const std::string* names = new std::string[3]{make(1), make(2), make(4)};
  const char* nm = names[P.tile >> 1].c_str();
  const int64_t lim = (int64_t)1 << 31;
  g.fast = g.a_m < lim && g.a_k < lim && g.b_k < lim && g.b_n < lim &&
           (128 * g.a_m + 16 * g.a_k) * (int64_t)sizeof(TA) < lim &&
           (64 * g.b_n + 16 * g.b_k) * (int64_t)sizeof(TB) < lim;
  g.tiles = P.tiles;
  const unsigned groups = (unsigned)((P.tiles + FILL_GROUP - 1) / FILL_GROUP) + g.fill_groups;
  const dim3 grid(g.fill_groups ? groups * FILL_GROUP : (unsigned)P.tiles);
  if (P.tile == 4)
    tlaunch(nm, P.flop, P.bytes, zgemm_grouped_kernel<Tc, TA, TB, TC, 4, 4, AK, BNC>, grid,
            dim3(256), s, g);
  else if (P.tile == 2)
    tlaunch(nm, P.flop, P.bytes, zgemm_grouped_kernel<Tc, TA, TB, TC, 2, 2, AK, BNC>, grid,
            dim3(256), s, g);
  else
    tlaunch(nm, P.flop, P.bytes, zgemm_grouped_kernel<Tc, TA, TB, TC, 1, 1, AK, BNC>, grid,
            dim3(256), s, g);
  PTN_LAUNCH_CHECK();
  return PTN_OK;
}

static size_t mpo_bytes(const Dims& D) { return (size_t)(D.Ml * D.d * D.d * D.Mr) * 16; }

// Zero fill of the n outputs: inside the first product's launch g, or (a caller's
// output that overlaps what that product or the mix reads) by zero_fill after the mix.
// in0, in1: the operands of the first product, w: the MPO tensor, each with its bytes.
static bool fill_with(GLaunch& g, void* out, int64_t n, const void* in0, size_t b0,
                      const void* in1, size_t b1, const void* w, size_t bw) {
  const char* o = (const char*)out;
  auto apart = [&](const void* p, size_t b) {
    return (const char*)p + b <= o || o + n * (int64_t)sizeof(double2) <= (const char*)p;
  };
  if (!apart(in0, b0) || !apart(in1, b1) || !apart(w, bw)) return false;
  g.fill = (double2*)out;
  g.nfill = n;
  g.fill_groups = (unsigned)((n + FILL_GROUP * FILL_PER_WG - 1) / (FILL_GROUP * FILL_PER_WG));
  return true;
}

// the sector mix of a plan: T2 (y) from T1 (x) with the MPO matrix w (complex128),
// complex128 operands in FP64 or complex64 in FP32 arithmetic; wtrans: w stored
// transposed (left environment)
template <int CAP>
static void mix_launch_cap(const SectorPlan* sp, bool fp64, int ni, int no, int64_t nr,
                           const void* w, const void* x, void* y, const int* skip, int wtrans,
                           hipStream_t s) {
  const dim3 grid((unsigned)sp->mix_tiles);
  const MixUnit* units = sp->dev_mix;
  const int nu = (int)sp->mix.size();
  if (fp64)
    tlaunch("k_mix_sectors<c128, c128>", 0.0, sp->mix_bytes * 16,
            k_mix_sectors<double2, double2, double, CAP>, grid, dim3(256), s, units, nu, ni, no,
            nr, (const double2*)w, (const double2*)x, (double2*)y, skip, wtrans);
  else
    tlaunch("k_mix_sectors<c64, c64>", 0.0, sp->mix_bytes * 8,
            k_mix_sectors<float2, float2, float, CAP>, grid, dim3(256), s, units, nu, ni, no, nr,
            (const double2*)w, (const float2*)x, (float2*)y, skip, wtrans);
}

static int mix_launch(const SectorPlan* sp, bool fp64, int ni, int no, int64_t nr, const void* w,
                      const void* x, void* y, const int* skip, int wtrans, hipStream_t s) {
  if (sp->mix_cap <= 8)
    mix_launch_cap<8>(sp, fp64, ni, no, nr, w, x, y, skip, wtrans, s);
  else if (sp->mix_cap <= 16)
    mix_launch_cap<16>(sp, fp64, ni, no, nr, w, x, y, skip, wtrans, s);
  else
    mix_launch_cap<MIX_LIST>(sp, fp64, ni, no, nr, w, x, y, skip, wtrans, s);
  PTN_LAUNCH_CHECK();
  return PTN_OK;
}

// H_eff through the grouped products: out = L^T . (W (x) (A . R)) as
// heff_apply computes it (same operand types: A and out complex128, L and R
// complex128 in FP64 and complex64 in FP32), only the blocks computed and out
// zero-filled outside them. Uses T1 and T2 of the heff_apply workspace.
int heff_apply_sectors(int prec, const Dims& D, const SectorPlan* sp, const void* l, int tl,
                       const void* w, const void* r, int tr, const void* a, void* out, void* ws,
                       size_t ws_bytes, hipStream_t s) {
  const int bp = grouped_prec(prec);
  if (!sp || bp < 0) return PTN_ERR_UNSUPPORTED;
  const int ct = bp == PTN_FP64 ? PTN_T_C128 : PTN_T_C64;
  if (tl != ct || tr != ct) return PTN_ERR_UNSUPPORTED;
  if (ws_bytes < heff_ws_bytes(prec, D)) return PTN_ERR_WORKSPACE;
  const size_t csz = bp == PTN_FP64 ? 16 : 8;
  const int64_t n1 = (D.Dl * D.d) * (D.Mr * D.Dr), nout = D.Dl * D.d * D.Dr;
  void* t1 = ws;   // written by the first product only inside its blocks (the mix reads no more)
  void* t2 = (char*)ws + (((size_t)n1 * csz + 255) & ~(size_t)255);
  const GBlock* b1 = sp->dev;
  const GBlock* b3 = sp->dev + sp->p1.blocks.size();
  const int* skip = skip_flag().p;
  int st;
  GLaunch g1{b1, (int)sp->p1.blocks.size(), D.d * D.Dr, 1, D.Mr * D.Dr, 1, D.d * D.Mr * D.Dr, 1,
             a, r, t1, skip, 0};
  const bool filled = fill_with(g1, out, nout, a, (size_t)nout * 16, r,
                                (size_t)(D.Dr * D.Mr * D.Dr) * csz, w, mpo_bytes(D));
  const int ni = (int)(D.d * D.Mr), no = (int)(D.Ml * D.d);
  if (bp == PTN_FP64) {
    if ((st = grouped_launch<double, double2, double2, double2, true, true>(g1, sp->p1, s)))
      return st;
    if ((st = mix_launch(sp, true, ni, no, D.Dr, w, t1, t2, skip, 0, s))) return st;
  } else {
    if ((st = grouped_launch<float, double2, float2, float2, true, true>(g1, sp->p1, s)))
      return st;
    if ((st = mix_launch(sp, false, ni, no, D.Dr, w, t1, t2, skip, 0, s))) return st;
  }
  PTN_LAUNCH_CHECK();
  if (!filled && (st = zero_fill<double2>(nout, out, s))) return st;
  GLaunch g3{b3, (int)sp->p3.blocks.size(), 1, D.Ml * D.Dl, D.Ml * D.d * D.Dr, 1, D.d * D.Dr, 1,
             l, t2, out, skip, 0};
  if (bp == PTN_FP64)
    return grouped_launch<double, double2, double2, double2, false, true>(g3, sp->p3, s);
  return grouped_launch<float, float2, float2, double2, false, true>(g3, sp->p3, s);
}

// Right environment step through the grouped products (env_right's chain:
// T1 = A . R, the mode mix, out = T2 . B^H), only the blocks computed and out
// zero-filled outside them. R has type tr (complex128 in FP64, complex64 in
// FP32); A, B and out are complex128. Uses T1 and T2 of the env workspace.
int env_right_sectors(int prec, const Dims& D, const SectorPlan* sp, const void* a, const void* b,
                      const void* w, const void* r, int tr, void* out, void* ws, size_t ws_bytes,
                      hipStream_t s) {
  const int bp = grouped_prec(prec);
  if (!sp || sp->kind != PLAN_ENV_RIGHT || bp < 0) return PTN_ERR_UNSUPPORTED;
  const int ct = bp == PTN_FP64 ? PTN_T_C128 : PTN_T_C64;
  if (tr != ct) return PTN_ERR_UNSUPPORTED;
  if (ws_bytes < env_ws_bytes(prec, D)) return PTN_ERR_WORKSPACE;
  const size_t csz = bp == PTN_FP64 ? 16 : 8;
  const size_t big = std::max((size_t)(D.Dl * D.d) * (size_t)(D.Mr * D.Dr),
                              (size_t)(D.Dl * D.Ml) * (size_t)(D.d * D.Dr)) * csz;
  void* t1 = ws;
  void* t2 = (char*)ws + ((big + 255) & ~(size_t)255);
  const GBlock* b1 = sp->dev;
  const GBlock* b3 = sp->dev + sp->p1.blocks.size();
  const int* skip = skip_flag().p;
  const int ni = (int)(D.d * D.Mr), no = (int)(D.Ml * D.d);
  int st;
  GLaunch g1{b1, (int)sp->p1.blocks.size(), D.d * D.Dr, 1, D.Mr * D.Dr, 1, D.d * D.Mr * D.Dr, 1,
             a, r, t1, skip, 0};
  // out[(l, m), lb] = sum T2[(l, m), (s', r')] conj(B[lb, (s', r')])
  GLaunch g3{b3, (int)sp->p3.blocks.size(), D.Ml * D.d * D.Dr, 1, 1, D.d * D.Dr, D.Ml * D.Dl, 1,
             t2, b, out, skip, 1};
  const int64_t nout = D.Dl * D.Ml * D.Dl;
  const bool filled = fill_with(g1, out, nout, a, (size_t)(D.Dl * D.d * D.Dr) * 16, r,
                                (size_t)(D.Dr * D.Mr * D.Dr) * csz, w, mpo_bytes(D));
  if (bp == PTN_FP64) {
    if ((st = grouped_launch<double, double2, double2, double2, true, true>(g1, sp->p1, s)))
      return st;
    if ((st = mix_launch(sp, true, ni, no, D.Dr, w, t1, t2, skip, 0, s))) return st;
    if (!filled && (st = zero_fill<double2>(nout, out, s))) return st;
    return grouped_launch<double, double2, double2, double2, true, false>(g3, sp->p3, s);
  }
  if ((st = grouped_launch<float, double2, float2, float2, true, true>(g1, sp->p1, s))) return st;
  if ((st = mix_launch(sp, false, ni, no, D.Dr, w, t1, t2, skip, 0, s))) return st;
  if (!filled && (st = zero_fill<double2>(nout, out, s))) return st;
  return grouped_launch<float, float2, double2, double2, true, false>(g3, sp->p3, s);
}

// Left environment step through the grouped products (env_left's chain:
// T1 = L . B*, the mode mix with the transposed MPO tensor, out = A^T . T2).
// L has type tl; A, B and out are complex128.
int env_left_sectors(int prec, const Dims& D, const SectorPlan* sp, const void* a, const void* b,
                     const void* w, const void* l, int tl, void* out, void* ws, size_t ws_bytes,
                     hipStream_t s) {
  const int bp = grouped_prec(prec);
  if (!sp || sp->kind != PLAN_ENV_LEFT || bp < 0) return PTN_ERR_UNSUPPORTED;
  const int ct = bp == PTN_FP64 ? PTN_T_C128 : PTN_T_C64;
  if (tl != ct) return PTN_ERR_UNSUPPORTED;
  if (ws_bytes < env_ws_bytes(prec, D)) return PTN_ERR_WORKSPACE;
  const size_t csz = bp == PTN_FP64 ? 16 : 8;
  const size_t big = std::max((size_t)(D.Dl * D.d) * (size_t)(D.Mr * D.Dr),
                              (size_t)(D.Dl * D.Ml) * (size_t)(D.d * D.Dr)) * csz;
  void* t1 = ws;
  void* t2 = (char*)ws + ((big + 255) & ~(size_t)255);
  const GBlock* b1 = sp->dev;
  const GBlock* b3 = sp->dev + sp->p1.blocks.size();
  const int* skip = skip_flag().p;
  const int ni = (int)(D.Ml * D.d), no = (int)(D.d * D.Mr);
  int st;
  // T1[(l, m), (s', r')] = sum_lb L[(l, m), lb] conj(B[lb, (s', r')])
  GLaunch g1{b1, (int)sp->p1.blocks.size(), D.Ml * D.Dl, 1, D.d * D.Dr, 1, D.Ml * D.d * D.Dr, 1,
             l, b, t1, skip, 1};
  // out[r, (m', r')] = sum_{(l, s)} A[(l, s), r] T2[(l, s), (m', r')]
  GLaunch g3{b3, (int)sp->p3.blocks.size(), 1, D.d * D.Dr, D.d * D.Mr * D.Dr, 1, D.Mr * D.Dr, 1,
             a, t2, out, skip, 0};
  const int64_t nout = D.Dr * D.Mr * D.Dr;
  const bool filled = fill_with(g1, out, nout, l, (size_t)(D.Dl * D.Ml * D.Dl) * csz, b,
                                (size_t)(D.Dl * D.d * D.Dr) * 16, w, mpo_bytes(D));
  if (bp == PTN_FP64) {
    if ((st = grouped_launch<double, double2, double2, double2, true, true>(g1, sp->p1, s)))
      return st;
    if ((st = mix_launch(sp, true, ni, no, D.Dr, w, t1, t2, skip, 1, s))) return st;
    if (!filled && (st = zero_fill<double2>(nout, out, s))) return st;
    return grouped_launch<double, double2, double2, double2, false, true>(g3, sp->p3, s);
  }
  if ((st = grouped_launch<float, float2, double2, float2, true, true>(g1, sp->p1, s))) return st;
  if ((st = mix_launch(sp, false, ni, no, D.Dr, w, t1, t2, skip, 1, s))) return st;
  if (!filled && (st = zero_fill<double2>(nout, out, s))) return st;
  return grouped_launch<float, double2, float2, double2, false, true>(g3, sp->p3, s);
}

}  // namespace ptn
