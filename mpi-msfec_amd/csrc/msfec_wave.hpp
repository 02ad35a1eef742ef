// Lane shifts, and sums over a wave and a workgroup.
#pragma once
#include <hip/hip_runtime.h>

namespace msfec_wave {

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// v of the lane to the right (left); zero at the ends of a row of 16 lanes
__device__ __forceinline__ double from_right(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x101, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x101, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double from_left(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x111, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x111, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// Block sums of 16 values per thread; thread t < 16 returns the t-th (red is
// free again after the caller's next barrier).  A wave sums them by halving:
// lanes 32, 16, 8 and 4 apart exchange half of what they hold (15 exchanges
// instead of 96), then the 4 lanes left with the same value add up.
template <int NW>
__device__ __forceinline__ double block_sums(const double* v, double (*red)[16]) {
  const int lane = threadIdx.x & 63;
  double a[8];
  int hi = lane >> 5 & 1;
#pragma unroll
  for (int k = 0; k < 8; ++k) a[k] = (hi ? v[8 + k] : v[k]) + __shfl_xor(hi ? v[k] : v[8 + k], 32);
  hi = lane >> 4 & 1;
#pragma unroll
  for (int k = 0; k < 4; ++k) a[k] = (hi ? a[4 + k] : a[k]) + __shfl_xor(hi ? a[k] : a[4 + k], 16);
  hi = lane >> 3 & 1;
#pragma unroll
  for (int k = 0; k < 2; ++k) a[k] = (hi ? a[2 + k] : a[k]) + __shfl_xor(hi ? a[k] : a[2 + k], 8);
  hi = lane >> 2 & 1;
  double s = (hi ? a[1] : a[0]) + __shfl_xor(hi ? a[0] : a[1], 4);
  s += __shfl_xor(s, 2);
  s += __shfl_xor(s, 1);
  __syncthreads();
  if ((lane & 3) == 0) red[threadIdx.x >> 6][lane >> 2] = s;
  __syncthreads();
  s = 0.0;
  if (threadIdx.x < 16)
#pragma unroll
    for (int i = 0; i < NW; ++i) s += red[i][threadIdx.x];
  return s;
}

}  // namespace msfec_wave
