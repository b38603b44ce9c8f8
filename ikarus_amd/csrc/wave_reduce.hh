// wave_reduce.hh — sums over the 64 lanes of a wavefront by DPP moves, a wait for loads, a short reciprocal.
//
// Shifts within rows of 16 lanes, then the row totals broadcast across rows; lane 63 ends with the total, read into a
// scalar register. A shuffle-based tree goes through the LDS crossbar at every step: a double's six steps take about
// 800 cycles there and 150 here, which is what the short vector kernels of a PCG iteration consist of.
#pragma once
#include <hip/hip_runtime.h>

namespace ik {

// v of another lane (0 where the move has no source lane or the row is not in ROWS)
template <int CTRL, int ROWS>
__device__ inline float dppMove(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROWS, 0xF, true));
}
template <int CTRL, int ROWS>
__device__ inline double dppMove(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, ROWS, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, ROWS, 0xF, true);
  return __builtin_bit_cast(double, (unsigned long long)(unsigned)hi << 32 | (unsigned)lo);
}
__device__ inline float lane63(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ inline double lane63(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo          = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, 63);
  const unsigned hi          = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), 63);
  return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}

// sum of v over the wavefront, the same in every lane; every lane must be active
template <typename T>
__device__ inline T waveSum(T v) {
  v += dppMove<0x111, 0xF>(v);  // row_shr:1
  v += dppMove<0x112, 0xF>(v);  // row_shr:2
  v += dppMove<0x114, 0xF>(v);  // row_shr:4
  v += dppMove<0x118, 0xF>(v);  // row_shr:8: lane 15 of each row has the row's sum
  v += dppMove<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
  v += dppMove<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
  return lane63(v);
}

// Waits for a loaded value here: the loads above it are in flight together, instead of each behind the branch or
// barrier that precedes its use
__device__ inline void arrived(double& v) { asm volatile("" : "+v"(v)); }
__device__ inline void arrived(int& v) { asm volatile("" : "+v"(v)); }
__device__ inline void arrived(float& v) { asm volatile("" : "+v"(v)); }
template <typename T, int N>
__device__ inline void arrived(T (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) arrived(v[i]);
}

// 1/d by the hardware estimate and two Newton steps: within an ulp of the division, at a third of its instructions
__device__ inline double reciprocal(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r        = fma(fma(-d, r, 1.0), r, r);
  return fma(fma(-d, r, 1.0), r, r);
}

}  // namespace ik
