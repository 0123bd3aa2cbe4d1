// The summaries of pages by 16-byte lanes, as a part of a launch: alone (page_minmax.hip) and with the
// rest of a prompt's cache (cache_init.hip).
#pragma once

#include "common.hpp"

namespace da {

// min/max that let NaN win, as torch.aminmax does.
__device__ __forceinline__ float nan_min(float m, float x) { return (x < m || x != x) ? x : m; }
__device__ __forceinline__ float nan_max(float m, float x) { return (x > m || x != x) ? x : m; }

template <typename T>
__device__ __forceinline__ u32x4 repack(const float *f);
template <>
__device__ __forceinline__ u32x4 repack<F32>(const float *f) {
  u32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = __builtin_bit_cast(uint32_t, f[i]);
  return v;
}
template <>
__device__ __forceinline__ u32x4 repack<F16>(const float *f) {
  u32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = pack_f16(f[2 * i], f[2 * i + 1]);
  return v;
}
template <>
__device__ __forceinline__ u32x4 repack<BF16>(const float *f) {
  u32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = pack_bf16(f[2 * i], f[2 * i + 1]);
  return v;
}

// Vector path: head_dim is a multiple of the 16-byte lane width and every stride keeps 16-byte
// alignment.  Items from `first` on, `n_threads` apart.
template <typename T>
__device__ __forceinline__ void page_minmax_vec(const char *__restrict__ k, int64_t head_stride, int64_t tok_stride,
                                                int n_heads, int64_t n_pages, int page, int chunks_per_row,
                                                char *__restrict__ out, int64_t first, int64_t n_threads) {
  constexpr int V = T::kVec;
  const int64_t items = n_pages * n_heads * chunks_per_row;
  for (int64_t it = first; it < items; it += n_threads) {
    const int c = (int)(it % chunks_per_row);
    const int64_t ph = it / chunks_per_row;
    const int h = (int)(ph % n_heads);
    const int64_t p = ph / n_heads;
    const char *src =
        k + (h * head_stride + p * page * tok_stride + (int64_t)c * V) * T::kBytes;
    float mn[V], mx[V], f[V];
    unpack<T>(load16(src), mn);
#pragma unroll
    for (int i = 0; i < V; ++i) mx[i] = mn[i];
    for (int t = 1; t < page; ++t) {
      unpack<T>(load16(src + (int64_t)t * tok_stride * T::kBytes), f);
#pragma unroll
      for (int i = 0; i < V; ++i) {
        mn[i] = nan_min(mn[i], f[i]);
        mx[i] = nan_max(mx[i], f[i]);
      }
    }
    const int64_t d = (int64_t)chunks_per_row * V;
    char *dst = out + (((int64_t)h * n_pages + p) * 2 * d + (int64_t)c * V) * T::kBytes;
    store16(dst, repack<T>(mn));
    store16(dst + d * T::kBytes, repack<T>(mx));
  }
}

inline bool minmax_vec_fits(const void *k, int64_t head_stride, int64_t tok_stride, int head_dim, int dtype, const void *out) {
  const int vec = 16 / elem_size(dtype);
  return head_dim % vec == 0 && head_stride % vec == 0 && tok_stride % vec == 0 && (uintptr_t)k % 16 == 0 &&
         (uintptr_t)out % 16 == 0;
}

}  // namespace da
