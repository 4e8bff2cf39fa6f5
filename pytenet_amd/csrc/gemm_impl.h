// Complex matrix products on CDNA4 MFMA through the real embedding
//   [Re C, Im C] = [Re A, Im A] . [[Re B, Im B], [-Im B, Re B]]
// i.e. a complex (M x N x K) product is a real (M x 2N x 2K) product whose A
// operand is the interleaved complex row itself and whose B operand is
// expanded from (Re B, Im B) when it is read from LDS. This keeps the
// interleaved complex layout of torch/NumPy in HBM, needs no extra flops
// (8 real flops per complex multiply-add, as four real products would) and
// uses one accumulator set per output tile.
//
// MFMA: v_mfma_f64_16x16x4f64 (FP64) and v_mfma_f32_16x16x4f32 (FP32) take
// A[i][k] in lane i + 16k and B[k][j] in lane j + 16k; the 16x16 result has
// column lane%16 and, in accumulator element v, row lane/16 + 4v (FP64) or
// row 4*(lane/16) + v (FP32).
#pragma once
#include <mutex>
#include <stdio.h>
#include <string.h>
#include <string>
#include <type_traits>
#include <unordered_map>
#include "common.h"

namespace ptn {

__device__ __forceinline__ d4_t mfma16(double a, double b, d4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4_t mfma16(float a, float b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
template <typename Tc> struct acc4;
template <> struct acc4<double> {
  typedef d4_t type;
  static __device__ __forceinline__ int row(int group, int v) { return group + 4 * v; }
  // lane group and accumulator element that hold a row
  static __device__ __forceinline__ int group(int row) { return row & 3; }
  static __device__ __forceinline__ int elem(int row) { return row >> 2; }
};
template <> struct acc4<float> {
  typedef f4_t type;
  static __device__ __forceinline__ int row(int group, int v) { return 4 * group + v; }
  static __device__ __forceinline__ int group(int row) { return row >> 2; }
  static __device__ __forceinline__ int elem(int row) { return row & 3; }
};

// A group of 4 waves (2 x 2) owns a BM x BN tile; each wave owns (16*TM) rows x
// (8*TN) complex columns. A workgroup holds WK such groups on the same tile,
// group w taking the w-th part of the k-stages; their sums are added in the
// order of the groups through LDS at the end. Splitting k inside the workgroup
// gives a product with few tiles more waves in flight and a shorter chain of
// dependent stages without a workspace or a second launch.
// BK complex k per LDS stage (BK / 4 steps of two MFMAs per tile); a group's LDS
// holds two stages (double buffer).
template <int TM, int TN, int BK_ = 8> struct TileCfg {
  static constexpr int WM = 16 * TM;
  static constexpr int WN = 8 * TN;
  static constexpr int BM = 2 * WM;
  static constexpr int BN = 2 * WN;
  static constexpr int BK = BK_;
  static constexpr int NA = BM * BK / 256;
  static constexpr int NB = BN * BK / 256;
};
// k-stage depth: FP32 stages twice as deep as FP64 ones (same LDS bytes), and the
// smallest tile twice as deep (256 threads stage at least one element each)
template <typename Tc, int TM> struct StageK {
  static constexpr int value = (TM == 1 || sizeof(Tc) == 4) ? 16 : 8;
};

struct GemmKArgs {
  int64_t M, N, K;
  const void* A; int64_t a_m, a_k; int conjA;
  const void* B; int64_t b_k, b_n; int conjB;
  void* C; int64_t c_m, c_n;
  int accumulate;
  int64_t bz_a, bz_b, bz_c;
  int tiles_n;          // number of column tiles
  int tiles_m;
  // optional block-sparsity masks (batch 1 only): bit t of word w of row tile
  // tm (column tile tn) is set when the A rows of tm (B columns of tn) have a
  // nonzero entry in k-stage 64 w + t; stages where the two masks do not
  // overlap contribute exactly zero and are skipped
  const uint64_t* maskA;
  const uint64_t* maskB;
  int mwords;
  // predication: the workgroups of batch problem z return at once when
  // skip[z * skip_stride] != 0
  const int* skip;
  int64_t skip_stride;
  // byte offsets inside a tile's operand rows fit 32 bits (launch_cfg)
  int fast;
};

// masked products keep their stage list in LDS: K / BK at most this many stages
constexpr int MAX_MASKED_STAGES = 2048;

// first k-stage >= from whose A and B masks overlap (every stage when unmasked)
__device__ __forceinline__ int next_stage(const GemmKArgs& g, int tm, int tn, int from, int nk) {
  if (!g.maskA) return from;
  for (int w = from >> 6; w < g.mwords; ++w) {
    uint64_t bits = g.maskA[(int64_t)tm * g.mwords + w] & g.maskB[(int64_t)tn * g.mwords + w];
    if (w == (from >> 6)) bits &= ~0ull << (from & 63);
    if (bits) {
      const int t = (w << 6) + __builtin_ctzll(bits);
      return t < nk ? t : nk;
    }
  }
  return nk;
}

// Tile masks of a GEMM operand. The operand has `ntile_items` items (A rows or
// B columns) split into tiles of `tile`, and K split into k-stages of `bk`;
// element (item, k) is at p[item * s_item + k * s_k] (+ batch 0 only).
// One workgroup per (tile, 64-stage word); threads walk the block along its
// contiguous dimension and OR the stage bits of nonzero entries in LDS.
template <typename T>
__global__ __launch_bounds__(256) void tile_mask_kernel(int64_t nitems, int64_t K, const T* __restrict__ p,
                                                        int64_t s_item, int64_t s_k, int tile, int bk,
                                                        int mwords, uint64_t* __restrict__ mask) {
  __shared__ unsigned int bits[2];
  const int tix = blockIdx.x, w = blockIdx.y;
  if (threadIdx.x < 2) bits[threadIdx.x] = 0;
  __syncthreads();
  const int64_t i0 = (int64_t)tix * tile;
  const int64_t k0 = (int64_t)w * 64 * bk;
  const int64_t ni = (i0 + tile < nitems ? i0 + tile : nitems) - i0;
  const int64_t nkk = (k0 + 64 * bk < K ? k0 + 64 * bk : K) - k0;
  const bool kfast = (s_k == 1) || (s_item != 1);
  unsigned int lo = 0, hi = 0;
  if (ni > 0 && nkk > 0) {
    for (int64_t e = threadIdx.x; e < ni * nkk; e += 256) {
      const int64_t it = kfast ? e / nkk : e % ni;
      const int64_t kk = kfast ? e % nkk : e / ni;
      const T v = p[(i0 + it) * s_item + (k0 + kk) * s_k];
      if (v.x != 0 || v.y != 0) {
        const int st = (int)(kk / bk);
        if (st < 32) lo |= 1u << st; else hi |= 1u << (st - 32);
      }
    }
  }
  if (lo) atomicOr(&bits[0], lo);
  if (hi) atomicOr(&bits[1], hi);
  __syncthreads();
  if (threadIdx.x == 0)
    mask[(int64_t)tix * mwords + w] = ((uint64_t)bits[1] << 32) | bits[0];
}

// bytes of mask workspace for an M x N x K product at any tile choice
inline size_t gemm_mask_bytes(int64_t M, int64_t N, int64_t K) {
  const int64_t words = ((K + 7) / 8 + 63) / 64;
  const int64_t tiles = (M + 63) / 64 + (N + 31) / 32;
  return (size_t)(tiles * words * 8 + 255) & ~(size_t)255;
}

// map the linear workgroup id so that the workgroups that run on one XCD
// (hardware assigns id % 8 to XCD id % 8) walk a contiguous range of tiles,
// column-tile fastest within a group of 8 row tiles, for L2 reuse of A and B.
__device__ __forceinline__ void tile_coords(int wg, int nwg, int tiles_m, int tiles_n, int& tm,
                                            int& tn) {
  int logical = wg;
  if ((nwg & 7) == 0) logical = (wg & 7) * (nwg >> 3) + (wg >> 3);
  const int group = 8;
  int per_group = group * tiles_n;
  int g = logical / per_group;
  int first_m = g * group;
  int rows = min(tiles_m - first_m, group);
  int in = logical - g * per_group;
  tm = first_m + in % rows;
  tn = in / rows;
}

// Operands are staged as whole complex elements, [k][row] and [k][column]. A step
// takes four complex k: lane group kk = lane / 16 holds complex k = 4 step + kk of
// its row of A and of its column of B, and one MFMA multiplies the real parts of
// A with (Re B | Im B), a second one the imaginary parts with (-Im B | Re B) for
// the (even | odd) real columns: the order of the real k inside a step is free as
// long as A and B agree, and this one reads every staged element once, as one
// LDS access, and needs no arithmetic on B but a select.
//
// What bounds it: FP64 MFMA issue on the large tile. The addresses of a stage
// are a uniform base plus a 32-bit offset per thread that is constant over the
// k-loop (rows and columns beyond the matrix are clamped to the last one: their
// results are not stored), so a stage's loads need no per-element address
// arithmetic and no predicates; only the last, partial k-stage and operands
// whose offsets exceed 32 bits take the general path.
template <typename Tc, typename TA, typename TB, typename TC, int TM, int TN, int WK,
          bool A_KCONTIG, bool B_NCONTIG>
__global__ __launch_bounds__(256 * WK) void zgemm_kernel(GemmKArgs g) {
  typedef TileCfg<TM, TN, StageK<Tc, TM>::value> T;
  constexpr int BM = T::BM, BN = T::BN, BK = T::BK, NA = T::NA, NB = T::NB;
  typedef typename acc4<Tc>::type acc_t;
  typedef typename cplx_of<Tc>::type C2;
  static_assert(NA >= 1 && NB >= 1, "a stage holds at least one element per thread");

  struct Stage {
    C2 A[2][BK][BM + 1];
    C2 B[2][BK][BN + 1];
  };
  __shared__ __align__(16) Stage stage_mem[WK];
  if (g.skip && g.skip[blockIdx.z * g.skip_stride]) return;

  const int grp = WK == 1 ? 0 : (int)(threadIdx.x >> 8);
  const int tid = threadIdx.x & 255;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm0 = (wave >> 1) * T::WM;
  const int wn0 = (wave & 1) * T::WN;
  auto& As = stage_mem[grp].A;
  auto& Bs = stage_mem[grp].B;

  int tm, tn;
  tile_coords(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * BM;
  const int64_t n0 = (int64_t)tn * BN;
  const int64_t bz = blockIdx.z;
  const TA* __restrict__ A = (const TA*)g.A + bz * g.bz_a + m0 * g.a_m;
  const TB* __restrict__ B = (const TB*)g.B + bz * g.bz_b + n0 * g.b_n;
  TC* __restrict__ C = (TC*)g.C + bz * g.bz_c;
  const Tc sa = g.conjA ? (Tc)-1 : (Tc)1;
  const Tc sb = g.conjB ? (Tc)-1 : (Tc)1;

  // element i of this thread in a stage: row / column (clamped) and k
  auto arow = [&](int i) -> int { return A_KCONTIG ? (tid + 256 * i) / BK : (tid + 256 * i) % BM; };
  auto ak = [&](int i) -> int { return A_KCONTIG ? (tid + 256 * i) % BK : (tid + 256 * i) / BM; };
  auto bcol = [&](int i) -> int { return B_NCONTIG ? (tid + 256 * i) % BN : (tid + 256 * i) / BK; };
  auto bk = [&](int i) -> int { return B_NCONTIG ? (tid + 256 * i) / BN : (tid + 256 * i) % BK; };
  const int mlast = (int)(g.M - m0 < BM ? g.M - m0 : BM) - 1;
  const int nlast = (int)(g.N - n0 < BN ? g.N - n0 : BN) - 1;
  uint32_t offa[NA], offb[NB];
#pragma unroll
  for (int i = 0; i < NA; ++i)
    offa[i] = (uint32_t)((min(arow(i), mlast) * g.a_m + ak(i) * g.a_k) * (int64_t)sizeof(TA));
#pragma unroll
  for (int i = 0; i < NB; ++i)
    offb[i] = (uint32_t)((min(bcol(i), nlast) * g.b_n + bk(i) * g.b_k) * (int64_t)sizeof(TB));

  // on the largest tile (one wave per SIMD) the elements stay as they were loaded until they
  // are staged, and the loads are kept ahead of the MFMAs (the compiler sinks them below else):
  // nothing else hides their latency. Environment step at D = 1024, MPO bond 8 (8192 x 2048 x 1024, c64 . c128):
  // 112 TFLOP/s, 78 without
  constexpr bool RAW = TM * TN >= 32;
  typename std::conditional<RAW, TA, C2>::type ra[NA];
  typename std::conditional<RAW, TB, C2>::type rb[NB];
  auto fetch = [](const auto* p, auto& v) {
    if constexpr (RAW) v = *p;
    else load_c<Tc>(p, v.x, v.y);
  };
  // stage at k0, all of it inside K, 32-bit offsets
  auto load_fast = [&](int64_t k0) {
    const char* Ak = (const char*)(A + k0 * g.a_k);
    const char* Bk = (const char*)(B + k0 * g.b_k);
#pragma unroll
    for (int i = 0; i < NA; ++i) fetch((const TA*)(Ak + offa[i]), ra[i]);
#pragma unroll
    for (int i = 0; i < NB; ++i) fetch((const TB*)(Bk + offb[i]), rb[i]);
    if constexpr (RAW) __builtin_amdgcn_sched_barrier(0);
  };
  // any stage (zeros beyond K)
  auto load_general = [&](int64_t k0) {
    const TA* Ak = A + k0 * g.a_k;
    const TB* Bk = B + k0 * g.b_k;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      ra[i] = {0, 0};
      if (k0 + ak(i) < g.K)
        fetch(Ak + (int64_t)min(arow(i), mlast) * g.a_m + (int64_t)ak(i) * g.a_k, ra[i]);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      rb[i] = {0, 0};
      if (k0 + bk(i) < g.K)
        fetch(Bk + (int64_t)min(bcol(i), nlast) * g.b_n + (int64_t)bk(i) * g.b_k, rb[i]);
    }
  };
  auto store_tiles = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NA; ++i) As[buf][ak(i)][arow(i)] = C2{(Tc)ra[i].x, sa * (Tc)ra[i].y};
#pragma unroll
    for (int i = 0; i < NB; ++i) Bs[buf][bk(i)][bcol(i)] = C2{(Tc)rb[i].x, sb * (Tc)rb[i].y};
  };

  acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

  const int l16 = lane & 15, kk = lane >> 4;
  const int pb = lane & 1;

  // k-stages to visit: a group's share [st0, st0 + per) of all of them, or (with
  // masks) those of its share where the A and B tile masks overlap, listed once
  // in LDS so that the main loop is a plain counted loop (keeps the accumulators
  // in place across iterations). The shares do not depend on the masks, so a
  // masked product adds in the order of the unmasked one. Every group runs
  // `iters` iterations (the barriers are the workgroup's).
  const int nk = (int)((g.K + BK - 1) / BK);
  __shared__ unsigned short stages[MAX_MASKED_STAGES];
  __shared__ int nstage_s[WK];
  const int per = (nk + WK - 1) / WK;
  const int st0 = grp * per, st1 = min(st0 + per, nk);
  int mine = max(0, st1 - st0), iters = per;
  if (g.maskA) {
    if (tid == 0) {
      int c = 0;
      for (int t = next_stage(g, tm, tn, st0, st1); t < st1;
           t = next_stage(g, tm, tn, t + 1, st1))
        stages[st0 + c++] = (unsigned short)t;
      nstage_s[grp] = c;
    }
    __syncthreads();
    mine = nstage_s[grp];
    iters = 0;
#pragma unroll
    for (int w = 0; w < WK; ++w) iters = max(iters, nstage_s[w]);
  }
  auto stage_of = [&](int it) -> int64_t {
    return g.maskA ? (int64_t)stages[st0 + it] : (int64_t)(st0 + it);
  };
  auto multiply = [&](int buf) {
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
  };
  // stage pipeline: global loads of the next stage into registers, MFMAs on
  // the current LDS buffer, registers into the other buffer, one barrier. The
  // first loop runs while the next stage is a whole one, without a branch in
  // its body.
  int buf = 0, it = 0;
  if (mine > 0) {
    load_general(stage_of(0) * BK);
    store_tiles(0);
  }
  __syncthreads();
  if (g.fast && !g.maskA) {
    // iterations whose next stage lies inside K, for every group
    const int nfast = min(per, (int)(g.K / BK) - (WK - 1) * per) - 1;
    for (; it < nfast; ++it) {
      load_fast((int64_t)(st0 + it + 1) * BK);
      multiply(buf);
      store_tiles(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
  }
  for (; it < iters; ++it) {
    const bool more = it + 1 < mine;
    if (more) load_general(stage_of(it + 1) * BK);
    if (it < mine) multiply(buf);
    if (more) store_tiles(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
  if constexpr (WK > 1) {
    // groups 1 .. WK - 1 hand their sums to group 0 through the stage buffers (one
    // row of tiles at a time), group 0 adds them in order and stores the tile
    constexpr int ROW = TN * 4 * 256;
    static_assert((WK - 1) * ROW * sizeof(Tc) <= sizeof(stage_mem), "sums fit the stage buffers");
    Tc* pool = (Tc*)&stage_mem[0];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (grp > 0) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            pool[(grp - 1) * ROW + (j * 4 + v) * 256 + tid] = acc[i][j][v];
      }
      __syncthreads();
      if (grp == 0) {
#pragma unroll
        for (int w = 1; w < WK; ++w)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              acc[i][j][v] += pool[(w - 1) * ROW + (j * 4 + v) * 256 + tid];
      }
      __syncthreads();
    }
    if (grp > 0) return;
  }

  // epilogue: lane holds the real (pb = 0) or imaginary (pb = 1) part of
  // complex column n for the rows of its accumulator elements v; the partner
  // lane (lane ^ 1) holds the other part. Even lanes store the rows of
  // elements 0, 1 and odd lanes those of elements 2, 3.
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      Tc mine_[4], other[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        mine_[v] = acc[i][j][v];
        other[v] = __shfl_xor(mine_[v], 1);
      }
      const int64_t n = n0 + wn0 + 8 * j + (l16 >> 1);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // constant register indices only (a lane-dependent index would force scratch)
        const int v = 2 * pb + h;
        const int64_t m = m0 + wm0 + 16 * i + acc4<Tc>::row(kk, v);
        double re = pb ? (double)other[2 + h] : (double)mine_[h];
        double im = pb ? (double)mine_[2 + h] : (double)other[h];
        if (m < g.M && n < g.N) {
          TC* p = C + m * g.c_m + n * g.c_n;
          if (g.accumulate) {
            double pr, pi;
            load_c<double>(p, pr, pi);
            re += pr; im += pi;
          }
          store_c(p, re, im);
        }
      }
    }
  }
}

// FP64 products of complex128 operands on the 128 x 64 and 64 x 32 tiles: the loop of
// zgemm_kernel with its stages loaded straight into LDS (global_load_lds of 16 bytes), three
// deep, and the fragments of the next half stage read before the MFMAs of the current one.
// Loads then need no registers and no LDS stores, stay in flight for two stages, and neither they
// nor the LDS reads are waited for between the MFMAs; one barrier per stage is placed between
// its halves. A wave's load writes 64 consecutive elements of LDS, so the layout follows from
// which element a lane fetches: [k][row] for operands contiguous in rows, else [row][k] with k
// exchanged by k ^ (row % 8), which keeps the 128-byte runs of the global reads and spreads the
// 16 rows that a fragment read touches over all banks. The sums are those of zgemm_kernel, in
// the same order. One array per stage and operand: the compiler then knows that a read does
// not wait for the loads in flight to the other stages.
// Bound by MFMA issue (84 % of the cycles busy before): 4096 x 5120 x 1024 64.6 -> 69.5 TFLOP/s,
// 2048^3 60.8 -> 68.8 (128 x 64); 1024 x 2560 x 512 54.7 -> 62.6 (64 x 32, two groups), 512 x
// 1024 x 2560 55.0 -> 62.9 (four groups).
template <int N, bool LGKM = false> __device__ __forceinline__ void wait_vm() {
  // s_waitcnt vmcnt(N), with LGKM also lgkmcnt(0)
  __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4 << 14) | 0x70 | (LGKM ? 0 : 0xF00));
}
__device__ __forceinline__ void wg_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
template <int WK_> struct LdsRing {
  static constexpr int WK = WK_;
};
template <typename Tc, typename TA, typename TB, typename TC, int TM, int TN, typename Ring,
          bool A_KCONTIG, bool B_NCONTIG>
__global__ __launch_bounds__(256 * Ring::WK) void zgemm_kernel(GemmKArgs g) {
  constexpr int WK = Ring::WK;
  static_assert(sizeof(Tc) == 8 && sizeof(TA) == 16 && sizeof(TB) == 16 && sizeof(TC) == 16,
                "FP64 products of complex128 operands");
  typedef TileCfg<TM, TN, 8> T;
  constexpr int BM = T::BM, BN = T::BN, BK = 8, NA = T::NA, NB = T::NB;
  __shared__ __align__(16) double2 A0[WK][BM * BK], A1[WK][BM * BK], A2[WK][BM * BK];
  __shared__ __align__(16) double2 B0[WK][BN * BK], B1[WK][BN * BK], B2[WK][BN * BK];
  if (g.skip && g.skip[blockIdx.z * g.skip_stride]) return;
  const int grp = WK == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int tid = threadIdx.x & 255, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave >> 1) * T::WM, wn0 = (wave & 1) * T::WN;
  int tm, tn;
  tile_coords(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN, bz = blockIdx.z;
  const char* A = (const char*)((const double2*)g.A + bz * g.bz_a + m0 * g.a_m);
  const char* B = (const char*)((const double2*)g.B + bz * g.bz_b + n0 * g.b_n);
  double2* __restrict__ C = (double2*)g.C + bz * g.bz_c;
  const int mlast = (int)(g.M - m0 < BM ? g.M - m0 : BM) - 1;
  const int nlast = (int)(g.N - n0 < BN ? g.N - n0 : BN) - 1;
  // element `lane` of chunk c (64 elements) of a stage: row / column and k
  auto arow = [&](int c) { return A_KCONTIG ? 8 * c + (lane >> 3) : 64 * (c % (BM / 64)) + lane; };
  auto ak = [&](int c) { return A_KCONTIG ? (lane & 7) ^ (lane >> 3) : c / (BM / 64); };
  auto bcol = [&](int c) { return B_NCONTIG ? (64 * c + lane) % BN : 8 * c + (lane >> 3); };
  auto bk = [&](int c) { return B_NCONTIG ? (64 * c + lane) / BN : (lane & 7) ^ (lane >> 3); };
  uint32_t offa[NA], offb[NB];
#pragma unroll
  for (int i = 0; i < NA; ++i)
    offa[i] = (uint32_t)((min(arow(wave * NA + i), mlast) * g.a_m + ak(wave * NA + i) * g.a_k) * 16);
#pragma unroll
  for (int i = 0; i < NB; ++i)
    offb[i] = (uint32_t)((min(bcol(wave * NB + i), nlast) * g.b_n + bk(wave * NB + i) * g.b_k) * 16);
  // the shares of k are those of zgemm_kernel: `per` of all stages to a group, the partial
  // last one to the group in whose share it lies; nst, mine, least: whole stages in all, of this
  // group and of the last one
  const int nst = (int)(g.K / BK), per = (int)((g.K + BK - 1) / BK + WK - 1) / WK;
  const int least = max(0, nst - (WK - 1) * per), most = min(per, nst);
  const int mine = WK == 1 ? nst : min(per, max(0, nst - grp * per));
  const int64_t sta = g.a_k * (BK * 16), stb = g.b_k * (BK * 16);
  const char* Ag = A + (int64_t)(mine ? grp * per : 0) * sta;
  const char* Bg = B + (int64_t)(mine ? grp * per : 0) * stb;
  typedef const __attribute__((address_space(1))) void* gp_t;
  typedef __attribute__((address_space(3))) void* lp_t;
  auto dma = [&](double2 (&As)[WK][BM * BK], double2 (&Bs)[WK][BN * BK], int st) {
    const int sc = max(min(st, mine - 1), 0);   // beyond the end: loaded again, not used
    const char* a = Ag + sc * sta;
    const char* b = Bg + sc * stb;
#pragma unroll
    for (int i = 0; i < NA; ++i)
      __builtin_amdgcn_global_load_lds((gp_t)(a + offa[i]), (lp_t)&As[grp][(wave * NA + i) * 64],
                                       16, 0, 0);
#pragma unroll
    for (int i = 0; i < NB; ++i)
      __builtin_amdgcn_global_load_lds((gp_t)(b + offb[i]), (lp_t)&Bs[grp][(wave * NB + i) * 64],
                                       16, 0, 0);
  };
  const int l16 = lane & 15, kk = lane >> 4, pb = lane & 1;
  // signs of the expanded B: conjugation of B in both, of A in the second one
  const uint32_t S = 0x80000000u;
  const uint32_t x0 = pb && g.conjB ? S : 0u, x1 = (pb || g.conjB ? 0u : S) ^ (g.conjA ? S : 0u);
  // fragments of the first half stage; the second half: k + 4 (k ^ 4 where k is exchanged)
  const int fa = A_KCONTIG ? (wm0 + l16) * 8 + (kk ^ (l16 & 7)) : kk * BM + wm0 + l16;
  const int nb = l16 >> 1;
  const int fb = B_NCONTIG ? kk * BN + wn0 + nb : (wn0 + nb) * 8 + (kk ^ nb);
  const int fa1 = A_KCONTIG ? fa ^ 4 : fa + 4 * BM, fb1 = B_NCONTIG ? fb + 4 * BN : fb ^ 4;
  constexpr int SA = A_KCONTIG ? 128 : 16, SB = B_NCONTIG ? 8 : 64;
  struct Frag {
    double2 a[TM], b[TN];
  };
  auto read = [&](const double2 (&As)[WK][BM * BK], const double2 (&Bs)[WK][BN * BK], int h,
                  Frag& f) {
    const double2* pa = &As[grp][h ? fa1 : fa];
    const double2* pbb = &Bs[grp][h ? fb1 : fb];
#pragma unroll
    for (int i = 0; i < TM; ++i) f.a[i] = pa[i * SA];
#pragma unroll
    for (int j = 0; j < TN; ++j) f.b[j] = pbb[j * SB];
  };
  d4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = d4_t{0, 0, 0, 0};
  auto flip = [](double v, uint32_t m) {
    const long long b = __double_as_longlong(v);
    return __longlong_as_double(((long long)((uint32_t)(b >> 32) ^ m) << 32) | (uint32_t)b);
  };
  auto mul = [&](const Frag& f) {
    double b0[TN], b1[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      b0[j] = flip(pb ? f.b[j].y : f.b[j].x, x0);
      b1[j] = flip(pb ? f.b[j].x : f.b[j].y, x1);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = mfma16(f.a[i].x, b0[j], acc[i][j]);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = mfma16(f.a[i].y, b1[j], acc[i][j]);
  };
  constexpr int VM = NA + NB;                      // loads of a stage
  auto sync = [&]() {
    wait_vm<VM, true>();
    wg_barrier();
  };
  Frag cur, nxt;
  auto step = [&](double2 (&As)[WK][BM * BK], double2 (&Bs)[WK][BN * BK],
                  double2 (&An)[WK][BM * BK], double2 (&Bn)[WK][BN * BK], int st, bool on) {
    read(As, Bs, 1, nxt);
    if (on) mul(cur);
    sync();             // stage st + 1 has landed and every wave has read stage st
    dma(As, Bs, st + 3);
    read(An, Bn, 0, cur);
    if (on) mul(nxt);
  };
  if (most > 0) {
    dma(A0, B0, 0);
    dma(A1, B1, 1);
    dma(A2, B2, 2);
    wait_vm<2 * VM>();
    wg_barrier();
    read(A0, B0, 0, cur);
    int st = 0;
    for (; st + 3 <= least; st += 3) {
      step(A0, B0, A1, B1, st, true);
      step(A1, B1, A2, B2, st + 1, true);
      step(A2, B2, A0, B0, st + 2, true);
    }
    for (; st < most; st += 3) {
      step(A0, B0, A1, B1, st, st < mine);
      if (st + 1 < most) step(A1, B1, A2, B2, st + 1, st + 1 < mine);
      if (st + 2 < most) step(A2, B2, A0, B0, st + 2, st + 2 < mine);
    }
    __builtin_amdgcn_s_waitcnt(0x70);   // no load may land in LDS from here on
  }
  __syncthreads();
  const int rem = (int)(g.K - (int64_t)nst * BK);
  if (rem) {   // the last, partial stage through registers
    const int64_t k0 = (int64_t)nst * BK;
    const int last = WK == 1 ? 0 : nst / per;
    if (grp == last) {
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        const int c = wave * NA + i;
        double2 v = make_double2(0.0, 0.0);
        if (ak(c) < rem)
          v = *(const double2*)(A + ((int64_t)min(arow(c), mlast) * g.a_m + (k0 + ak(c)) * g.a_k) * 16);
        A0[grp][c * 64 + lane] = v;
      }
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int c = wave * NB + i;
        double2 v = make_double2(0.0, 0.0);
        if (bk(c) < rem)
          v = *(const double2*)(B + ((int64_t)min(bcol(c), nlast) * g.b_n + (k0 + bk(c)) * g.b_k) * 16);
        B0[grp][c * 64 + lane] = v;
      }
    }
    __syncthreads();
    if (grp == last) {
      read(A0, B0, 0, cur);
      read(A0, B0, 1, nxt);
      mul(cur);
      mul(nxt);
    }
    __syncthreads();
  }
  if constexpr (WK > 1) {
    constexpr int ROW = TN * 4 * 256;
    static_assert(ROW * 8 <= sizeof(A0), "a group's sums fit an operand buffer");
    double* pool[3] = {(double*)&A0[0][0], (double*)&A1[0][0], (double*)&A2[0][0]};
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int w = 1; w < WK; ++w)
        if (grp == w) {
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) pool[w - 1][(j * 4 + v) * 256 + tid] = acc[i][j][v];
        }
      __syncthreads();
      if (grp == 0) {
#pragma unroll
        for (int w = 1; w < WK; ++w)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[i][j][v] += pool[w - 1][(j * 4 + v) * 256 + tid];
      }
      __syncthreads();
    }
    if (grp > 0) return;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      double mine_[4], other[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        mine_[v] = acc[i][j][v];
        other[v] = __shfl_xor(mine_[v], 1);
      }
      const int64_t n = n0 + wn0 + 8 * j + (l16 >> 1);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int v = 2 * pb + h;
        const int64_t m = m0 + wm0 + 16 * i + acc4<double>::row(kk, v);
        double re = pb ? other[2 + h] : mine_[h];
        double im = pb ? mine_[2 + h] : other[h];
        if (m < g.M && n < g.N) {
          double2* p = C + m * g.c_m + n * g.c_n;
          if (g.accumulate) {
            re += p->x;
            im += p->y;
          }
          *p = make_double2(re, im);
        }
      }
    }
}

// The smallest products. A workgroup of WK waves owns 16 rows x (8*TN) complex
// columns and every wave takes its part of k: a product of a few thousand
// outputs then reaches all CUs, which the 2 x 2-wave tiles above do not (64 x 256
// outputs are 8 workgroups of 64 x 32), and its chain of dependent MFMAs is
// K / (4 WK) steps long. A lane loads the complex elements that it feeds to the
// MFMAs straight from global memory (16 rows x 4 k of A, 4 k x 8 columns of B per
// step: whole 64- or 128-byte runs in either order of the operands), U steps
// ahead of their use; there is no staging and no barrier in the loop. The WK
// partial tiles are added in the order of the waves through LDS.
template <int TN_> struct WaveTile {
  static constexpr int TN = TN_;
  static constexpr int BM = 16;
  static constexpr int BN = 8 * TN_;
};
template <typename Tc, typename TA, typename TB, typename TC, typename Tile, int WK,
          bool A_KCONTIG, bool B_NCONTIG>
__global__ __launch_bounds__(64 * WK) void zgemm_kernel(GemmKArgs g) {
  constexpr int TN = Tile::TN, BM = Tile::BM, BN = Tile::BN;
  constexpr int U = 4;                       // steps per batch of loads
  typedef typename acc4<Tc>::type acc_t;
  typedef typename cplx_of<Tc>::type C2;
  __shared__ __align__(16) Tc red[WK][TN * 4][64];
  if (g.skip && g.skip[blockIdx.z * g.skip_stride]) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, kk = lane >> 4, pb = lane & 1;
  int tm, tn;
  tile_coords(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int64_t bz = blockIdx.z;
  const Tc sa = g.conjA ? (Tc)-1 : (Tc)1;
  const Tc sb = g.conjB ? (Tc)-1 : (Tc)1;
  const TA* __restrict__ A = (const TA*)g.A + bz * g.bz_a + min(m0 + l16, g.M - 1) * g.a_m;
  const TB* __restrict__ B[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j)
    B[j] = (const TB*)g.B + bz * g.bz_b + min(n0 + 8 * j + (l16 >> 1), g.N - 1) * g.b_n;
  // steps of four k; this wave's are [s0, s1)
  const int nstep = (int)((g.K + 3) / 4);
  const int per = (nstep + WK - 1) / WK;
  const int s0 = wave * per, s1 = min(s0 + per, nstep);

  acc_t acc[TN][2];
#pragma unroll
  for (int j = 0; j < TN; ++j) acc[j][0] = acc[j][1] = acc_t{0, 0, 0, 0};
  struct Batch {
    C2 a[U], b[U][TN];
  };
  // steps s .. s + U - 1, k clamped to the last one; a step beyond s1 is not used
  auto load = [&](int s, Batch& q) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t k = min((int64_t)4 * (s + u) + kk, g.K - 1);
      load_c<Tc>(A + k * g.a_k, q.a[u].x, q.a[u].y);
#pragma unroll
      for (int j = 0; j < TN; ++j) load_c<Tc>(B[j] + k * g.b_k, q.b[u][j].x, q.b[u][j].y);
    }
  };
  auto multiply = [&](int s, const Batch& q) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s + u < s1) {
        const bool in = (int64_t)4 * (s + u) + kk < g.K;
        const Tc ar = in ? q.a[u].x : Tc(0), ai = in ? sa * q.a[u].y : Tc(0);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const Tc br = in ? q.b[u][j].x : Tc(0), bi = in ? sb * q.b[u][j].y : Tc(0);
          acc[j][0] = mfma16(ar, pb ? bi : br, acc[j][0]);
          acc[j][1] = mfma16(ai, pb ? br : -bi, acc[j][1]);
        }
      }
    }
  };
  if (s0 < s1) {
    Batch q0, q1;
    load(s0, q0);
    for (int s = s0; s < s1; s += 2 * U) {
      load(s + U, q1);
      multiply(s, q0);
      if (s + U < s1) {
        load(s + 2 * U, q0);
        multiply(s + U, q1);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave][j * 4 + v][lane] = acc[j][0][v] + acc[j][1][v];
  __syncthreads();
  // one complex output per thread: its real part sits in an even lane of the
  // result layout, the imaginary part in the next one
  TC* __restrict__ C = (TC*)g.C + bz * g.bz_c;
  for (int e = threadIdx.x; e < BM * BN; e += 64 * WK) {
    const int r = e / BN, c = e % BN;
    const int64_t m = m0 + r, n = n0 + c;
    if (m >= g.M || n >= g.N) continue;
    const int src = acc4<Tc>::group(r) * 16 + 2 * (c & 7);
    const int slot = (c >> 3) * 4 + acc4<Tc>::elem(r);
    double re = 0, im = 0;
#pragma unroll
    for (int w = 0; w < WK; ++w) {
      re += (double)red[w][slot][src];
      im += (double)red[w][slot][src + 1];
    }
    TC* p = C + m * g.c_m + n * g.c_n;
    if (g.accumulate) {
      double pr, pi;
      load_c<double>(p, pr, pi);
      re += pr;
      im += pi;
    }
    store_c(p, re, im);
  }
}

// algorithmic work of one product launch: 8 real flops per complex
// multiply-add; bytes = each operand once, C written (and read if accumulating)
inline double gemm_flop(const ZGemm& z) {
  return 8.0 * (double)z.M * (double)z.N * (double)z.K * (double)z.batch;
}
template <typename TA, typename TB, typename TC>
inline double gemm_bytes(const ZGemm& z) {
  return (double)z.batch * ((double)z.M * z.K * sizeof(TA) + (double)z.K * z.N * sizeof(TB) +
                            (double)z.M * z.N * sizeof(TC) * (z.accumulate ? 2 : 1));
}
// kernel instance name as a profiler lists it (template arguments, without
// the namespace and the argument list), e.g.
// zgemm_kernel<float, c64, c64, c128, 4, 8, 1, true, true> (TM = 0: the wave tile)
template <typename Tc, typename TA, typename TB, typename TC, int TM, int TN, int WK = 1>
inline const char* gemm_kernel_name(bool ak, bool bn, const char* kernel = "zgemm_kernel") {
  static std::mutex mu;
  static std::unordered_map<std::string, std::string> names;
  char buf[160];
  // the split-bf16 kernel has no compute-type and no k-group argument
  const bool with_tc = strcmp(kernel, "zgemm_kernel") == 0;
  char tile[32], wk[16] = "";
  if (TM > 0) snprintf(tile, sizeof(tile), "%d, %d", TM, TN);
  else snprintf(tile, sizeof(tile), "WaveTile<%d>", TN);
  if (with_tc) snprintf(wk, sizeof(wk), "%d, ", WK);
  snprintf(buf, sizeof(buf), "%s<%s%s%s, %s, %s, %s, %s%s, %s>", kernel,
           with_tc ? type_tag<Tc>::s : "", with_tc ? ", " : "", type_tag<TA>::s,
           type_tag<TB>::s, type_tag<TC>::s, tile, wk, ak ? "true" : "false",
           bn ? "true" : "false");
  std::lock_guard<std::mutex> lk(mu);
  auto it = names.find(buf);
  if (it == names.end()) it = names.emplace(buf, buf).first;
  return it->second.c_str();
}

// masks for the chosen tile shape (BM rows of A, BN columns of B, BK-wide
// k-stages) in `mws` (gemm_mask_bytes bytes), batch 1 only
template <typename TA, typename TB>
inline int build_masks(const ZGemm& z, GemmKArgs& g, int BM, int BN, int BK, void* mws,
                       size_t mws_bytes, hipStream_t s) {
  g.maskA = nullptr; g.maskB = nullptr; g.mwords = 0;
  if (!mws || z.batch != 1 || z.K == 0) return PTN_OK;
  const int64_t nk = (z.K + BK - 1) / BK;
  if (nk > MAX_MASKED_STAGES) return PTN_OK;   // dense product (correct, no skipping)
  const int words = (int)((nk + 63) / 64);
  const size_t need = (size_t)((int64_t)g.tiles_m + g.tiles_n) * words * 8;
  // the workspace is sized for 64 x 32 tiles; the masks of a short product on smaller
  // tiles may not fit it: no skipping then, the result is the same
  if (mws_bytes < need) return PTN_OK;
  uint64_t* ma = (uint64_t*)mws;
  uint64_t* mb = ma + (int64_t)g.tiles_m * words;
  tile_mask_kernel<TA><<<dim3((unsigned)g.tiles_m, (unsigned)words), 256, 0, s>>>(
      z.M, z.K, (const TA*)z.A, z.a_m, z.a_k, BM, BK, words, ma);
  tile_mask_kernel<TB><<<dim3((unsigned)g.tiles_n, (unsigned)words), 256, 0, s>>>(
      z.N, z.K, (const TB*)z.B, z.b_n, z.b_k, BN, BK, words, mb);
  PTN_LAUNCH_CHECK();
  g.maskA = ma; g.maskB = mb; g.mwords = words;
  return PTN_OK;
}

// kernel arguments of a product on BM x BN tiles; false if the grid is too large
inline bool fill_args(const ZGemm& z, GemmKArgs& g, int BM, int BN) {
  g.M = z.M; g.N = z.N; g.K = z.K;
  g.A = z.A; g.a_m = z.a_m; g.a_k = z.a_k; g.conjA = z.conjA;
  g.B = z.B; g.b_k = z.b_k; g.b_n = z.b_n; g.conjB = z.conjB;
  g.C = z.C; g.c_m = z.c_m; g.c_n = z.c_n;
  g.accumulate = z.accumulate;
  g.bz_a = z.bz_a; g.bz_b = z.bz_b; g.bz_c = z.bz_c;
  g.tiles_m = (int)((z.M + BM - 1) / BM);
  g.tiles_n = (int)((z.N + BN - 1) / BN);
  g.maskA = nullptr; g.maskB = nullptr; g.mwords = 0;
  g.skip = skip_flag().p;
  g.skip_stride = skip_flag().stride;
  g.fast = 0;
  return (int64_t)g.tiles_m * g.tiles_n <= 0x7fffffff && z.batch <= 65535;
}

// launch of the kernel instance for the operands' contiguity: a K-contiguous A
// when its k stride is 1 (or K == 1), else M-contiguous; B alike
#define PTN_GEMM_LAUNCH(nm, z, g, s, threads, ...)                                              \
  do {                                                                                          \
    const bool ak_ = (z.a_k == 1) || (z.a_m != 1), bn_ = (z.b_n == 1) || (z.b_k != 1);          \
    const dim3 grid_((unsigned)((int64_t)g.tiles_m * g.tiles_n), 1, (unsigned)z.batch);         \
    const double fl_ = gemm_flop(z), by_ = gemm_bytes<TA, TB, TC>(z);                           \
    if (ak_ && bn_)                                                                             \
      tlaunch(nm(true, true), fl_, by_, zgemm_kernel<Tc, TA, TB, TC, __VA_ARGS__, true, true>,  \
              grid_, dim3(threads), s, g);                                                      \
    else if (ak_)                                                                               \
      tlaunch(nm(true, false), fl_, by_,                                                        \
              zgemm_kernel<Tc, TA, TB, TC, __VA_ARGS__, true, false>, grid_, dim3(threads), s,  \
              g);                                                                               \
    else if (bn_)                                                                               \
      tlaunch(nm(false, true), fl_, by_,                                                        \
              zgemm_kernel<Tc, TA, TB, TC, __VA_ARGS__, false, true>, grid_, dim3(threads), s,  \
              g);                                                                               \
    else if constexpr (sizeof(Tc) == 8)                                                         \
      tlaunch(nm(false, false), fl_, by_,                                                       \
              zgemm_kernel<Tc, TA, TB, TC, __VA_ARGS__, false, false>, grid_, dim3(threads), s, \
              g);                                                                               \
    else                                                                                        \
      return PTN_ERR_UNSUPPORTED;   /* no reduced-precision product has this layout */          \
    PTN_LAUNCH_CHECK();                                                                         \
    return PTN_OK;                                                                              \
  } while (0)

inline int64_t tiles_of(const ZGemm& z, int BM, int BN) {
  return ((z.M + BM - 1) / BM) * ((z.N + BN - 1) / BN) * z.batch;
}

// loads of 16 bytes into LDS need operands on 16-byte boundaries
inline bool dma_operands(const ZGemm& z) { return (((uintptr_t)z.A | (uintptr_t)z.B) & 15) == 0; }
template <int TM, int TN, int WK>
inline int launch_dma(const ZGemm& z, const GemmKArgs& g, hipStream_t s) {
  const bool ak = (z.a_k == 1) || (z.a_m != 1), bn = (z.b_n == 1) || (z.b_k != 1);
  const dim3 grid((unsigned)((int64_t)g.tiles_m * g.tiles_n), 1, (unsigned)z.batch);
  const double fl = gemm_flop(z), by = gemm_bytes<double2, double2, double2>(z);
  auto go = [&](auto a, auto b) {
    static const std::string nm =
        "zgemm_kernel<double, c128, c128, c128, " + std::to_string(TM) + ", " +
        std::to_string(TN) + ", LdsRing<" + std::to_string(WK) + ">, " +
        (a.value ? "true" : "false") + ", " + (b.value ? "true" : "false") + ">";
    tlaunch(nm.c_str(), fl, by,
            zgemm_kernel<double, double2, double2, double2, TM, TN, LdsRing<WK>, a.value, b.value>,
            grid, dim3(256 * WK), s, g);
  };
  using Y = std::true_type;
  using N = std::false_type;
  if (ak && bn) go(Y(), Y());
  else if (ak) go(Y(), N());
  else if (bn) go(N(), Y());
  else go(N(), N());
  PTN_LAUNCH_CHECK();
  return PTN_OK;
}

template <typename Tc, typename TA, typename TB, typename TC, int TM, int TN, int WK = 1>
inline int launch_cfg(const ZGemm& z, hipStream_t s, void* mws = nullptr, size_t mws_bytes = 0) {
  typedef TileCfg<TM, TN, StageK<Tc, TM>::value> T;
  GemmKArgs g;
  if (!fill_args(z, g, T::BM, T::BN)) return PTN_ERR_ARG;
  const int64_t lim = (int64_t)1 << 31;   // non-negative strides with offsets below 2 GiB
  g.fast = z.a_m >= 0 && z.a_k >= 0 && z.b_k >= 0 && z.b_n >= 0 && z.a_m < lim && z.a_k < lim &&
           z.b_k < lim && z.b_n < lim &&
           (T::BM * z.a_m + T::BK * z.a_k) * (int64_t)sizeof(TA) < lim &&
           (T::BN * z.b_n + T::BK * z.b_k) * (int64_t)sizeof(TB) < lim;
  int st = build_masks<TA, TB>(z, g, T::BM, T::BN, T::BK, mws, mws_bytes, s);
  if (st) return st;
  if constexpr (sizeof(Tc) == 8 && TM >= 2) {
    static_assert(sizeof(TA) == 16 && sizeof(TB) == 16 && sizeof(TC) == 16, "complex128 operands");
    // At most two whole stages leave nothing to keep in flight, and with more tiles than the chip
    // holds with three stage buffers each the two of the register-staged kernel let more of them in:
    // 1095 x 2249 x 5 (1278 tiles of 64 x 32) 12.3 -> 10.6 us, 8000 x 500 x 3 15.8 -> 14.1, 4000 x 3000 x 5
    // (1504 of 128 x 64) 42.1 -> 39.0; from K = 24 on the ring is as fast or faster.
    const int64_t fit = 256 * (160 * 1024 / (3 * (T::BM + T::BN) * T::BK * (int64_t)sizeof(TA)));
    const bool brief = WK == 1 && z.K < 3 * T::BK && tiles_of(z, T::BM, T::BN) > fit;
    if (g.fast && !g.maskA && dma_operands(z) && !brief) return launch_dma<TM, TN, WK>(z, g, s);
  }
  auto nm = [](bool ak, bool bn) {   // formatted once per instance
    static const char* const n[4] = {gemm_kernel_name<Tc, TA, TB, TC, TM, TN, WK>(false, false),
                                     gemm_kernel_name<Tc, TA, TB, TC, TM, TN, WK>(false, true),
                                     gemm_kernel_name<Tc, TA, TB, TC, TM, TN, WK>(true, false),
                                     gemm_kernel_name<Tc, TA, TB, TC, TM, TN, WK>(true, true)};
    return n[2 * ak + bn];
  };
  PTN_GEMM_LAUNCH(nm, z, g, s, 256 * WK, TM, TN, WK);
}

// the wave-tile kernel for the smallest products
template <typename Tc, typename TA, typename TB, typename TC, int TN, int WK>
inline int launch_wave(const ZGemm& z, hipStream_t s) {
  typedef WaveTile<TN> T;
  GemmKArgs g;
  if (!fill_args(z, g, T::BM, T::BN)) return PTN_ERR_ARG;
  auto nm = [](bool ak, bool bn) {
    static const char* const n[4] = {gemm_kernel_name<Tc, TA, TB, TC, 0, TN, WK>(false, false),
                                     gemm_kernel_name<Tc, TA, TB, TC, 0, TN, WK>(false, true),
                                     gemm_kernel_name<Tc, TA, TB, TC, 0, TN, WK>(true, false),
                                     gemm_kernel_name<Tc, TA, TB, TC, 0, TN, WK>(true, true)};
    return n[2 * ak + bn];
  };
  PTN_GEMM_LAUNCH(nm, z, g, s, 64 * WK, T, WK);
}

// opt-in autotuning of the tile shape (ptn_set_autotune): set once per process
bool autotune_enabled();

// Tile choice, from the times of every configuration over shapes M, N, K = 16 ..
// 5120 (FP64 figures, us or TFLOP/s at M x N x K):
//  * at most 320 outputs tiles of 16 x 8: one wave tile per CU or so. The product is
//    latency-bound and the wave kernel is the shortest chain (64 x 256 x 320: 6.0 us
//    against 11.3 of the next best; 128 x 256 x 640: 9.1 against 18.5; equal at
//    200 x 400 x 1000 = 650 tiles); below K = 192 four waves have work enough.
//  * large tiles (128 x 64; FP32 also 128 x 128) where their number fills whole waves
//    of two workgroups per CU: full waves 69.2 TFLOP/s against 67.0 of 64 x 32 tiles
//    (1024 x 4096 x 5120), but 53.6 against 62.3 with 640 tiles in 512 slots
//    (5120 x 1024 x 2048, without the loads into LDS). FP32: 128 x 128 down to 0.8 of a wave's
//    slots.
//  * 64 x 32 tiles from 192 up. Fewer than about two per CU leave the matrix cores
//    waiting for operands: then k is split over two or four groups of the workgroup
//    (256 tiles, 512 x 1024 x 2560: 50.1 / 61.8 / 62.9 TFLOP/s with 1 / 2 / 4 groups).
//    FP64, loaded into LDS: two groups pay up to 2048 tiles (1280 tiles, 1024 x 2560 x 512: 59.7 /
//    62.6 / 56.9; 2048, 2048^3: 66.0 / 66.4; 10240: 67.2 / 66.5). Staged through registers (all
//    of FP32) one group does from 600 on (FP64, 1280 tiles: 59.0 / 55.9 / 51.2); masked or unaligned FP64
//    products, which are staged so too, still take the groups of the others. Batches in
//    FP64 take one group from 256 tiles on unless k is long (24 of 100 x 200 x 500, 336 tiles: 85 us with
//    four groups, 77 with one; 64 of 128 x 320 x 64, 1280 tiles: 37 with two, 30 with one; 4 of 100 x 1000 x
//    200, 256 tiles: 19 and 20; 4 of 240 x 960 x 2000, 480 tiles: four are no slower).
//  * tile-skipping products (mask workspace given) never take the large tiles: the
//    small one skips the zero blocks of sector-structured operands at finer
//    granularity, which outweighs its lower efficiency per flop (U(1) two-site DMRG
//    at L=128, D=2048: 76 s against 82 s per sweep).
//  * the split of k depends on shape and type alone (k_groups), so that masked and
//    unmasked products add in the same order.
//  * 32 x 16 tiles for fewer, or where 64-row tiles would be a third padding (the
//    32-row products of the blocked QR, 32 x 1984 x 248 x 8: 27.8 us against 42.2).
inline double wave_fill(int64_t tiles, int64_t slots) {
  return (double)tiles / (double)((tiles + slots - 1) / slots * slots);
}
inline bool wave_tile_product(const ZGemm& z) { return tiles_of(z, 16, 8) <= 320; }
// 128 x 128 tiles (FP32), 128 x 64 tiles, 64 x 32 tiles (else 32 x 16)
template <typename Tc> inline bool wide_tiles(const ZGemm& z) {
  const int64_t wide = tiles_of(z, 128, 128);
  return sizeof(Tc) == 4 && wide >= 512 && wave_fill(wide, 512) >= 0.8;
}
inline bool large_tiles(const ZGemm& z) {
  const int64_t t44 = tiles_of(z, 128, 64);
  return t44 >= 512 && wave_fill(t44, 512) >= 0.96;
}
inline bool medium_tiles(const ZGemm& z) {   // tiles of 32 x 16 per one of 64 x 32: 4 without padding
  const int64_t t22 = tiles_of(z, 64, 32);
  return t22 >= 192 && 3 * t22 <= tiles_of(z, 32, 16);
}
// groups of k of a product beyond the wave tiles
template <typename Tc> inline int k_groups(const ZGemm& z) {
  if (z.K < 64 || wide_tiles<Tc>(z) || large_tiles(z)) return 1;
  if (!medium_tiles(z)) return tiles_of(z, 32, 16) >= 512 ? 1 : z.K < 256 ? 2 : 4;
  const int64_t t22 = tiles_of(z, 64, 32);
  if (t22 >= (sizeof(Tc) == 8 ? 2048 : 600)) return 1;
  if (sizeof(Tc) == 8 && z.batch > 1 && t22 >= 256 && z.K <= 1024) return 1;
  return z.K < 256 || t22 >= 600 ? 2 : 4;
}

template <typename Tc, typename TA, typename TB, typename TC>
inline int launch_heuristic(const ZGemm& z, hipStream_t s, void* mws, size_t mws_bytes) {
  if (wave_tile_product(z)) {
    if (z.K >= 192) return launch_wave<Tc, TA, TB, TC, 1, 8>(z, s);
    return launch_wave<Tc, TA, TB, TC, 1, 4>(z, s);
  }
  const bool masked = mws && z.batch == 1;
  if constexpr (sizeof(Tc) == 4)
    if (!masked && wide_tiles<Tc>(z)) return launch_cfg<Tc, TA, TB, TC, 4, 8>(z, s);
  if (!masked && large_tiles(z)) return launch_cfg<Tc, TA, TB, TC, 4, 4>(z, s);
  const int groups = k_groups<Tc>(z);
  if (medium_tiles(z)) {
    if (groups == 1) return launch_cfg<Tc, TA, TB, TC, 2, 2>(z, s, mws, mws_bytes);
    if (groups == 2) return launch_cfg<Tc, TA, TB, TC, 2, 2, 2>(z, s, mws, mws_bytes);
    return launch_cfg<Tc, TA, TB, TC, 2, 2, 4>(z, s, mws, mws_bytes);
  }
  if (groups == 1) return launch_cfg<Tc, TA, TB, TC, 1, 1>(z, s, mws, mws_bytes);
  if (groups == 2) return launch_cfg<Tc, TA, TB, TC, 1, 1, 2>(z, s, mws, mws_bytes);
  return launch_cfg<Tc, TA, TB, TC, 1, 1, 4>(z, s, mws, mws_bytes);
}

template <typename Tc, typename TA, typename TB, typename TC>
inline int launch_choice(int c, const ZGemm& z, hipStream_t s) {
  if (c == 0) return launch_heuristic<Tc, TA, TB, TC>(z, s, nullptr, 0);
  if (c == 1) return launch_cfg<Tc, TA, TB, TC, 2, 2>(z, s);
  if (c == 2) return launch_cfg<Tc, TA, TB, TC, 4, 4>(z, s);
  if constexpr (sizeof(Tc) == 4) return launch_cfg<Tc, TA, TB, TC, 4, 8>(z, s);
  return PTN_ERR_ARG;
}

// Tile autotuner: the first product of a given shape (M, N, K, batch and the
// contiguity of the operands) times the rule's choice and the other large tiles (two timed
// launches each after one untimed, HIP events on the caller's stream) and
// keeps the fastest for that shape. It synchronises the stream once per new shape, hence opt-in.
// Tuned are products that overwrite C (a repeated launch then leaves the same result) and
// for which the rule takes a single group of k: the candidates are single groups, and
// with the division of k the sums are the same in every tile, so that the
// result does not depend on what was timed.
template <typename Tc, typename TA, typename TB, typename TC>
inline int launch_tuned(const ZGemm& z, hipStream_t s) {
  struct Key {
    int64_t M, N, K, batch, flags;
    bool operator==(const Key& o) const {
      return M == o.M && N == o.N && K == o.K && batch == o.batch && flags == o.flags;
    }
  };
  struct Hash {
    size_t operator()(const Key& k) const {
      return std::hash<int64_t>()(k.M * 1000003 ^ k.N * 10007 ^ k.K * 101 ^ k.batch * 7 ^ k.flags);
    }
  };
  static std::mutex mu;
  static std::unordered_map<Key, int, Hash> best;
  const Key key{z.M, z.N, z.K, z.batch,
                (int64_t)(z.a_k == 1) | (int64_t)(z.a_m == 1) << 1 | (int64_t)(z.b_n == 1) << 2 |
                    (int64_t)(z.b_k == 1) << 3};
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = best.find(key);
    if (it != best.end()) return launch_choice<Tc, TA, TB, TC>(it->second, z, s);
  }
  const int nc = sizeof(Tc) == 4 ? 4 : 3;
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess) return PTN_ERR_HIP;
  if (hipEventCreate(&e1) != hipSuccess) { (void)hipEventDestroy(e0); return PTN_ERR_HIP; }
  int bestc = 0, st = PTN_OK;
  float bestms = 0.0f;
  for (int c = 0; c < nc && st == PTN_OK; ++c) {
    if ((st = launch_choice<Tc, TA, TB, TC>(c, z, s))) break;
    (void)hipEventRecord(e0, s);
    for (int r = 0; r < 2 && st == PTN_OK; ++r) st = launch_choice<Tc, TA, TB, TC>(c, z, s);
    (void)hipEventRecord(e1, s);
    if (hipEventSynchronize(e1) != hipSuccess) { st = PTN_ERR_HIP; break; }
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    if (c == 0 || ms < bestms) { bestms = ms; bestc = c; }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (st) return st;
  {
    std::lock_guard<std::mutex> lk(mu);
    best[key] = bestc;
  }
  // C holds the last configuration's (identical) result; write it once more
  // with the chosen one so that the output never depends on tuning order
  return launch_choice<Tc, TA, TB, TC>(bestc, z, s);
}

template <typename Tc, typename TA, typename TB, typename TC>
inline int launch_typed(const ZGemm& z, hipStream_t s, void* mws = nullptr, size_t mws_bytes = 0) {
  if (mws && z.batch == 1) return launch_heuristic<Tc, TA, TB, TC>(z, s, mws, mws_bytes);
  // (the wave tile is not in question for the products that the rule gives it)
  if (!z.accumulate && autotune_enabled() && !noalloc_mode() && !wave_tile_product(z) &&
      k_groups<Tc>(z) == 1) {
    // tuning synchronises the stream, which a stream capture does not allow
    hipStreamCaptureStatus cst = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cst) == hipSuccess && cst == hipStreamCaptureStatusNone)
      return launch_tuned<Tc, TA, TB, TC>(z, s);
  }
  return launch_heuristic<Tc, TA, TB, TC>(z, s, mws, mws_bytes);
}

}  // namespace ptn
