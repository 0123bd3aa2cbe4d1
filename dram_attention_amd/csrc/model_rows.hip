// Row-wise parts of the Llama-shaped model around the attention layers, for many rows
// (a prompt): RMS norm with the residual addition in front of it, rotary embedding of the
// projected queries and keys, and the SwiGLU product.  Counterparts of RMSNorm,
// apply_rotary_emb and FeedForward.forward of the reference's model
// (evaluation/dram-attention/model.py:66-78, :126-136, :236-245).
//
// Bound: HBM.  Each kernel reads every operand once and writes every result once, 16 bytes
// per lane; torch's operators made 6 passes for a norm, 9 for a rotation (most of them in
// fp32) and 2 for the product.  Results are rounded where the torch operators they stand
// for round: fp32 inside, the type T between.
//
// Measured at 8192 rows of dim 4096, hidden 14336, 32/8 heads of 128, bf16: norm 25 us, with
// the addition in front 40 us; rotation of queries and keys 32 us (168 MB, 5.3 TB/s); SwiGLU
// product 105 us (705 MB, 6.7 TB/s).  A prompt of 8192 tokens through two layers: 9.33 -> 7.48 ms;
// a token through four layers from Python, 200 -> 72 launches: 2.35 -> 1.38 ms.
#include "model_math.hpp"

namespace da {

constexpr int kRowThreads = 256;

// One row per group of kLanes lanes (64 or the whole block), kept in registers.
template <typename T, int kVecs, int kLanes>
__global__ void __launch_bounds__(kRowThreads)
rms_norm_kernel(const char *__restrict__ x, const char *__restrict__ add, char *__restrict__ sum_out,
                const char *__restrict__ weight, float eps, char *__restrict__ out, int64_t rows, int dim) {
  constexpr int kPerBlock = kRowThreads / kLanes;
  const int64_t row = (int64_t)blockIdx.x * kPerBlock + threadIdx.x / kLanes;
  const int lane = threadIdx.x % kLanes;
  const int vecs = dim / T::kVec;
  const bool live = row < rows;
  const int64_t base = (live ? row : rows - 1) * (int64_t)dim * T::kBytes;
  float f[kVecs][T::kVec];
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < kVecs; ++u) {
    const int j = lane + u * kLanes;
    if (j < vecs) {
      unpack<T>(load16(x + base + (int64_t)j * 16), f[u]);
      if (add != nullptr) {
        float g[T::kVec];
        unpack<T>(load16(add + base + (int64_t)j * 16), g);
#pragma unroll
        for (int i = 0; i < T::kVec; ++i) f[u][i] = round_to<T>(f[u][i] + g[i]);
        if (live) store16(sum_out + base + (int64_t)j * 16, pack_vec<T>(f[u]));
      }
      ss += sum_of_squares<T>(f[u]);
    }
  }
  ss = group_sum<64>(ss);
  if constexpr (kLanes > 64) {
    __shared__ float part[kRowThreads / 64];
    if (threadIdx.x % 64 == 0) part[threadIdx.x / 64] = ss;
    __syncthreads();
    static_assert(kRowThreads / 64 == 4, "the waves' sums in pairs");
    ss = (part[0] + part[1]) + (part[2] + part[3]);
  }
  const float inv = rms_scale(ss, dim, eps);
#pragma unroll
  for (int u = 0; u < kVecs; ++u) {
    const int j = lane + u * kLanes;
    if (j < vecs && live) {
      float w[T::kVec];
      unpack<T>(load16(weight + (int64_t)j * 16), w);
#pragma unroll
      for (int i = 0; i < T::kVec; ++i) f[u][i] = round_to<T>(f[u][i] * inv) * w[i];
      store16(out + base + (int64_t)j * 16, pack_vec<T>(f[u]));
    }
  }
}

// 16 bytes of a query or key row per lane, rotated in place; the table's row of a token
// (fp32 cosine and sine per channel pair) is shared by its heads and comes from cache.
template <typename T>
__global__ void __launch_bounds__(kRowThreads)
rope_rows_kernel(char *__restrict__ q, int64_t q_tok_b, char *__restrict__ k, int64_t k_tok_b, int q_vecs,
                 int k_vecs, int row_vecs, const float *__restrict__ table, int64_t rows) {
  const int per_tok = q_vecs + k_vecs;
  const int64_t j = (int64_t)blockIdx.x * kRowThreads + threadIdx.x;
  if (j >= rows * per_tok) return;
  const int64_t tok = j / per_tok;
  const int within = (int)(j % per_tok);
  char *p = within < q_vecs ? q + tok * q_tok_b + (int64_t)within * 16
                            : k + tok * k_tok_b + (int64_t)(within - q_vecs) * 16;
  const int chunk = (within < q_vecs ? within : within - q_vecs) % row_vecs;   // within the head
  const float *cs = table + (tok * row_vecs + chunk) * T::kVec;   // (cos, sin) per pair
  float f[T::kVec], r[T::kVec];
  unpack<T>(load16(p), f);
#pragma unroll
  for (int i = 0; i < T::kVec; i += 4) *(float4 *)(r + i) = *(const float4 *)(cs + i);
#pragma unroll
  for (int i = 0; i < T::kVec; i += 2) rotate_pair(f[i], f[i + 1], r[i], r[i + 1]);
  store16(p, pack_vec<T>(f));
}

template <typename T>
__global__ void __launch_bounds__(kRowThreads)
swiglu_kernel(const char *gate, const char *up, char *out, int64_t vecs) {   // (out may be gate or up)
  const int64_t j = (int64_t)blockIdx.x * kRowThreads + threadIdx.x;
  if (j >= vecs) return;
  float a[T::kVec], b[T::kVec];
  unpack<T>(load16_stream(gate + j * 16), a);
  unpack<T>(load16_stream(up + j * 16), b);
#pragma unroll
  for (int i = 0; i < T::kVec; ++i) a[i] = round_to<T>(silu<T>(a[i])) * b[i];
  store16(out + j * 16, pack_vec<T>(a));
}

template <typename T>
static int launch_rms_norm(const char *x, const char *add, char *sum_out, const char *weight, float eps, char *out,
                           int64_t rows, int dim, hipStream_t s) {
  const int vecs = dim / T::kVec;
  // Rows of up to 128 vectors (1024 elements of 16 bits) are a wave's; longer ones a block's.
#define DA_NORM(v, lanes)                                                                                   \
  hipLaunchKernelGGL((rms_norm_kernel<T, v, lanes>), dim3((unsigned)ceil_div(rows, kRowThreads / lanes)),   \
                     dim3(kRowThreads), 0, s, x, add, sum_out, weight, eps, out, rows, dim)
  if (vecs <= 128) DA_NORM(2, 64);
  else if (vecs <= 512) DA_NORM(2, 256);
  else if (vecs <= 1024) DA_NORM(4, 256);
  else DA_NORM(8, 256);
#undef DA_NORM
  return launch_status("da_rms_norm");
}

}  // namespace da

extern "C" int da_rms_norm(const void *x, const void *add, void *sum_out, const void *weight, float eps, void *out,
                           int64_t rows, int dim, int dtype, void *stream) {
  using namespace da;
  DA_REQUIRE(rows >= 0 && dim > 0, "da_rms_norm: bad shape");
  DA_REQUIRE(dtype == DA_F32 || dtype == DA_F16 || dtype == DA_BF16, "da_rms_norm: unknown dtype %d", dtype);
  if (rows == 0) return DA_OK;
  DA_REQUIRE(x && weight && out && (!add == !sum_out), "da_rms_norm: null pointer");
  const int64_t row_bytes = (int64_t)dim * elem_size(dtype);
  if (row_bytes % 16 != 0 || row_bytes > 8 * 256 * 16 || rows > 0x7fffffff)
    return fail(DA_ENOTSUP, "da_rms_norm: rows of a multiple of 16 bytes up to 32 KiB (got %lld)",
                (long long)row_bytes);
  DA_REQUIRE(((uintptr_t)x | (uintptr_t)add | (uintptr_t)sum_out | (uintptr_t)weight | (uintptr_t)out) % 16 == 0,
             "da_rms_norm: operands must be 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  const char *xb = (const char *)x, *ab = (const char *)add, *wb = (const char *)weight;
  if (dtype == DA_BF16) return launch_rms_norm<BF16>(xb, ab, (char *)sum_out, wb, eps, (char *)out, rows, dim, s);
  if (dtype == DA_F16) return launch_rms_norm<F16>(xb, ab, (char *)sum_out, wb, eps, (char *)out, rows, dim, s);
  return launch_rms_norm<F32>(xb, ab, (char *)sum_out, wb, eps, (char *)out, rows, dim, s);
}

extern "C" int da_rope_rows(void *q, int64_t q_tok_stride, void *k, int64_t k_tok_stride, int n_q_heads,
                            int n_kv_heads, int head_dim, const float *table, int64_t rows, int dtype,
                            void *stream) {
  using namespace da;
  DA_REQUIRE(rows >= 0 && n_q_heads >= 0 && n_kv_heads >= 0 && head_dim > 0, "da_rope_rows: bad shape");
  DA_REQUIRE(dtype == DA_F32 || dtype == DA_F16 || dtype == DA_BF16, "da_rope_rows: unknown dtype %d", dtype);
  const int e = elem_size(dtype);
  if (rows == 0 || n_q_heads + n_kv_heads == 0) return DA_OK;
  DA_REQUIRE(table && (q || !n_q_heads) && (k || !n_kv_heads), "da_rope_rows: null pointer");
  if (head_dim * e % 16 != 0)
    return fail(DA_ENOTSUP, "da_rope_rows: head rows of a multiple of 16 bytes (got %d)", head_dim * e);
  DA_REQUIRE(q_tok_stride * e % 16 == 0 && k_tok_stride * e % 16 == 0 &&
                 ((uintptr_t)q | (uintptr_t)k | (uintptr_t)table) % 16 == 0,
             "da_rope_rows: operands must be 16-byte aligned");
  const int row_vecs = head_dim * e / 16;
  const int64_t items = rows * (n_q_heads + n_kv_heads) * row_vecs;
  if (ceil_div(items, kRowThreads) > 0x7fffffff) return fail(DA_ENOTSUP, "da_rope_rows: too many rows");
  const dim3 grid((unsigned)ceil_div(items, kRowThreads));
  hipStream_t s = (hipStream_t)stream;
#define DA_ROPE(T)                                                                                               \
  hipLaunchKernelGGL((rope_rows_kernel<T>), grid, dim3(kRowThreads), 0, s, (char *)q, q_tok_stride *e, (char *)k, \
                     k_tok_stride *e, n_q_heads *row_vecs, n_kv_heads *row_vecs, row_vecs, table, rows)
  if (dtype == DA_BF16) DA_ROPE(BF16);
  else if (dtype == DA_F16) DA_ROPE(F16);
  else DA_ROPE(F32);
#undef DA_ROPE
  return launch_status("da_rope_rows");
}

extern "C" int da_swiglu(const void *gate, const void *up, void *out, int64_t n, int dtype, void *stream) {
  using namespace da;
  DA_REQUIRE(n >= 0, "da_swiglu: negative length");
  DA_REQUIRE(dtype == DA_F32 || dtype == DA_F16 || dtype == DA_BF16, "da_swiglu: unknown dtype %d", dtype);
  if (n == 0) return DA_OK;
  DA_REQUIRE(gate && up && out, "da_swiglu: null pointer");
  const int64_t bytes = n * elem_size(dtype);
  if (bytes % 16 != 0 || ceil_div(bytes / 16, kRowThreads) > 0x7fffffff)
    return fail(DA_ENOTSUP, "da_swiglu: a multiple of 16 bytes (got %lld)", (long long)bytes);
  DA_REQUIRE(((uintptr_t)gate | (uintptr_t)up | (uintptr_t)out) % 16 == 0,
             "da_swiglu: operands must be 16-byte aligned");
  const dim3 grid((unsigned)ceil_div(bytes / 16, kRowThreads));
  hipStream_t s = (hipStream_t)stream;
#define DA_SWIGLU(T)                                                                                         \
  hipLaunchKernelGGL((swiglu_kernel<T>), grid, dim3(kRowThreads), 0, s, (const char *)gate, (const char *)up, \
                     (char *)out, bytes / 16)
  if (dtype == DA_BF16) DA_SWIGLU(BF16);
  else if (dtype == DA_F16) DA_SWIGLU(F16);
  else DA_SWIGLU(F32);
#undef DA_SWIGLU
  return launch_status("da_swiglu");
}
