// Wavefront sums shared by the SOR and MG kernels (device code).
#pragma once

#include <hip/hip_runtime.h>

namespace pgamd {

// v of the lane a DPP control selects (within a row of 16 lanes)
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false),
                          __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false));
}

// Sum over each row of 16 lanes, the same bits in every lane of the row: partners 1 and 2 apart in a quad, then the
// mirrored halves of 8 and of 16 lanes (each step adds the same two operands in every lane of a pair, only commuted).
template <typename T>
__device__ __forceinline__ T row_sum(T v) {
  v = v + dpp<0xB1>(v);    // quad [1,0,3,2]
  v = v + dpp<0x4E>(v);    // quad [2,3,0,1]
  v = v + dpp<0x141>(v);   // half-row mirror
  return v + dpp<0x140>(v);   // row mirror
}

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane), __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Sum over the wavefront: rows of 16 lanes as above, then (r0 + r1) + (r2 + r3) from scalar registers, so every lane gets
// the same bits.
template <typename T>
__device__ __forceinline__ T wave_sum_dpp(T v) {
  v = row_sum(v);
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

// Sum of v[0..N-1] as a tree over adjacent halves.
template <int N, typename T>
__device__ __forceinline__ T tree_sum(const T* v) {
  if constexpr (N == 1)
    return v[0];
  else
    return tree_sum<N / 2>(v) + tree_sum<N - N / 2>(v + N / 2);
}

// Butterfly sum over the wavefront (partners 32, 16, ... 1 apart); with lanes beyond a shorter segment at zero, the bits
// of the butterfly over that segment.
__device__ __forceinline__ float wave_sum_butterfly(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

}  // namespace pgamd
