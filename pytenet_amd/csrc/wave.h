// Scalar operations over one wave in registers, shared by the QR, Jacobi and
// Lanczos kernels.
#pragma once
#include "common.h"

namespace ptn {

// sum over the wave, in every lane: rotations inside the rows of 16 lanes (DPP), then the
// four row sums read as scalars (an exchange through LDS per step takes several
// times as long)
template <int CTRL> __device__ __forceinline__ double dpp_rot(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double lane_value(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double wave_sum(double v) {
  v += dpp_rot<0x128>(v);   // row rotate right by 8, 4, 2, 1
  v += dpp_rot<0x124>(v);
  v += dpp_rot<0x122>(v);
  v += dpp_rot<0x121>(v);
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

// 1 / sqrt(x) to full double precision for normal positive x: the hardware's estimate
// (relative error about 2^-24) and one third-order step. Chains of
// dependent operations (plane rotations) set the speed of its callers; the library's rsqrt,
// sqrt and division take several times as many.
__device__ __forceinline__ double rsq_full(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// sum over each row of 16 lanes, in every lane of it
__device__ __forceinline__ double row_sum(double v) {
  v += dpp_rot<0x128>(v);   // row rotate right by 8, 4, 2, 1
  v += dpp_rot<0x124>(v);
  v += dpp_rot<0x122>(v);
  v += dpp_rot<0x121>(v);
  return v;
}
// barrier that orders LDS accesses only: stores to memory that only the threads which
// made them read back stay in flight across it
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

}  // namespace ptn
