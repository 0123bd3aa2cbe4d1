// Arithmetic that the row-wise kernels of the model (model_rows.hip) and its one-row
// linear layers (decode_linear.hip) share, so that a prompt and a decode step round alike.
#pragma once
#include "common.hpp"

namespace da {

template <typename T>
__device__ __forceinline__ u32x4 pack_vec(const float *f);
template <>
__device__ __forceinline__ u32x4 pack_vec<BF16>(const float *f) {
  return u32x4{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]), pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7])};
}
template <>
__device__ __forceinline__ u32x4 pack_vec<F16>(const float *f) {
  return u32x4{pack_f16(f[0], f[1]), pack_f16(f[2], f[3]), pack_f16(f[4], f[5]), pack_f16(f[6], f[7])};
}
template <>
__device__ __forceinline__ u32x4 pack_vec<F32>(const float *f) {
  return u32x4{__builtin_bit_cast(uint32_t, f[0]), __builtin_bit_cast(uint32_t, f[1]),
               __builtin_bit_cast(uint32_t, f[2]), __builtin_bit_cast(uint32_t, f[3])};
}

__device__ __forceinline__ float rms_scale(float sum_of_squares, int dim, float eps) {
  return rsqrtf(sum_of_squares / (float)dim + eps);
}

// (even, odd) turned by the angle whose cosine and sine are c and s.
__device__ __forceinline__ void rotate_pair(float &even, float &odd, float c, float s) {
  const float e = even * c - odd * s, o = even * s + odd * c;
  even = e;
  odd = o;
}

// x / (1 + exp(-x)); for the 16-bit types the hardware exponential and reciprocal (each
// within an ulp or two of fp32), which the rounding of the result swallows.  The reciprocal
// is taken of a sixteenth: v_rcp_f32 gives zero for 1 / d below 2^-126, i.e. for x between
// -88.7 and -87.3, where x / d is still a normal number of the type.
template <typename T>
__device__ __forceinline__ float silu(float x) {
  const float d = 1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x);
  return (x * 0.0625f) * __builtin_amdgcn_rcpf(d * 0.0625f);
}
template <>
__device__ __forceinline__ float silu<F32>(float x) { return x / (1.f + expf(-x)); }

}  // namespace da
