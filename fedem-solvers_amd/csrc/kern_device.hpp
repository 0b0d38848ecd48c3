// Device code that several kernel files use.
#pragma once
#include "kernels.hpp"

namespace fgpu {

using f64x4 = __attribute__((__vector_size__(4 * sizeof(double)))) double;

static inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

// Workgroups of a launch are dispatched round-robin over the eight XCDs of
// the MI355X (workgroup b on XCD b mod 8), each with its own L2.  Both maps from
// workgroup b to a task are bijections of [0, n).
//
// xcd_ranges: every XCD takes one contiguous range of the task list, so that
// neighbouring tasks, which share panel columns or source rows, share an L2.
__device__ __forceinline__ int xcd_ranges(int b, int n) {
  const int q = n >> 3, r = n & 7, c = b & 7, m = b >> 3;
  return c < r ? c * (q + 1) + m : r * (q + 1) + (c - r) * q + m;
}
// xcd_fours: neighbouring tasks go to one XCD by fours, the fours round the
// XCDs, for lists whose tasks get shorter or longer along the list.
__device__ __forceinline__ int xcd_fours(int b, int n) {
  constexpr int G = 4;
  if (b >= n / (8 * G) * (8 * G)) return b;
  const int c = b & 7, m = b >> 3;
  return ((m / G) * 8 + c) * G + m % G;
}

// Value of v in lane src (uniform src), through the scalar unit: no LDS
// round trip and no memory wait between the broadcasts of a sweep.
__device__ __forceinline__ double lane_bcast(double v, int src) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), src);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), src);
  return __hiloint2double(hi, lo);
}

// 1/d to rounding: the hardware estimate r0 (relative error e below 2^-20)
// and r0 (1 + e + e^2).
__device__ __forceinline__ double recip64(double d) {
  const double r = __builtin_amdgcn_rcp(d), e = __builtin_fma(-d, r, 1.0);
  return __builtin_fma(__builtin_fma(e, e, e), r, r);
}

}  // namespace fgpu
