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

// Of one 16-byte vector, in pairs: what a lane adds up one after the other is then a few vectors.
template <typename T>
__device__ __forceinline__ float sum_of_squares(const float *f) {
  float s[T::kVec / 2];
#pragma unroll
  for (int i = 0; i < T::kVec / 2; ++i) s[i] = fmaf(f[2 * i], f[2 * i], f[2 * i + 1] * f[2 * i + 1]);
#pragma unroll
  for (int n = T::kVec / 4; n >= 1; n /= 2)
#pragma unroll
    for (int i = 0; i < n; ++i) s[i] += s[i + n];
  return s[0];
}

// 1 / sqrt(mean + eps): the hardware's root with one Newton step, its residual 1 - v r^2
// formed by fused multiply-adds.  Without the step, and with all squares of a lane in one
// chain, the fp32 norm is 4-6 % further from float64 than torch's operators (5.2-5.3e-8 against
// 5.0e-8 in the 2-norm).
__device__ __forceinline__ float rms_scale(float sum_of_squares, int dim, float eps) {
  const float v = sum_of_squares / (float)dim + eps;
  const float r = rsqrtf(v);
  const float h = v * r;
  const float e = fmaf(-fmaf(v, r, -h), r, fmaf(-h, r, 1.f));
  return e == e ? fmaf(0.5f * r, e, r) : r;   // (v of 0, infinity or NaN: as the root gives it)
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
