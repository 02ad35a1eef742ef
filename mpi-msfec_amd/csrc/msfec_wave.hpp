// Buffer loads, lane shifts, sums over a wave and a workgroup, the inverse root.
#pragma once
#include <hip/hip_runtime.h>

namespace msfec_wave {

// `bytes` bytes at p, the same for all lanes, for buffer loads: a load outside
// of them returns zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const double* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(p), 0, bytes, 0x00027000);
}
// The value at byte offset `lane` (per lane) + `uni` (uniform).  With plain
// pointers the compiler forms a 64-bit address per lane for every load of an
// unrolled loop ahead of it, and spills them.
typedef unsigned buffer_v2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double buffer_f64(__amdgpu_buffer_rsrc_t b, int lane, int uni) {
  const buffer_v2 t = __builtin_amdgcn_raw_buffer_load_b64(b, lane, uni, 0);
  return __hiloint2double((int)t.y, (int)t.x);
}
__device__ __forceinline__ void buffer_f64(__amdgpu_buffer_rsrc_t b, int lane, int uni, double v) {
  const buffer_v2 t = {(unsigned)__double2loint(v), (unsigned)__double2hiint(v)};
  __builtin_amdgcn_raw_buffer_store_b64(t, b, lane, uni, 0);
}

// Sum over the N lanes (a power of two, at most 16) of a row, or of N values
// that repeat within it: every lane has it, in the same bits, as a + b = b + a.
template <int N>
__device__ __forceinline__ double row_sum(double v) {
#define MSFEC_ROR(k)                                                                         \
  if constexpr (N > k)                                                                       \
    v += __hiloint2double(                                                                   \
        __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x120 + k, 0xf, 0xf, false),       \
        __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x120 + k, 0xf, 0xf, false))
  MSFEC_ROR(8);
  MSFEC_ROR(4);
  MSFEC_ROR(2);
  MSFEC_ROR(1);
#undef MSFEC_ROR
  return v;
}
__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// Sum over a wave, in every lane: by moves within the rows of 16 lanes and
// scalar registers.  (The exchanges of __shfl_xor go through the LDS unit, six
// round trips one after the other.  A pass of the CG kernels: 64 cells of 16^3
// with tensors 1.71 ms with those, 1.58 ms so; 3-D RT_DQ, 64 cells, 3.79 and
// 3.53 ms.)
__device__ __forceinline__ double wave_sum(double v) {
  v = row_sum<16>(v);
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}
// Sum of the NW values at red (one of each wave), in every lane.
template <int NW>
__device__ __forceinline__ double waves_sum(const double* red) {
  static_assert(NW <= 16, "one row");
  return row_sum<NW>(red[threadIdx.x & (NW - 1)]);
}

// x^-1/2 for x > 0: the instruction and two Newton steps, the last one as a
// correction of the value, which leaves about one rounding (y (1.5 - x y^2 / 2)
// leaves three: the bases of the band solver were off by 1.04e-15 to 1.91e-14
// instead of 8.6e-16 to 1.58e-14 then, 5 % to 20 % more than with divisions; a
// step takes as long)
__device__ __forceinline__ double inv_sqrt(double x) {
  double y = __builtin_amdgcn_rsq(x);
  y = y * fma(-0.5 * x * y, y, 1.5);
  return fma(0.5 * y, fma(-x * y, y, 1.0), y);
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
