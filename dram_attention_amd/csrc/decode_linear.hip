// The linear layers of the Llama-shaped model for ONE token (a decode step): y = W x with
// W (N, K) row-major, with the step's small operations folded in where their operands
// already are:
//   in front   RMS norm of the input row (every workgroup norms the row it is about to use:
//              8 KB from cache, behind its first weight loads)
//   behind     rotary embedding of the query and key rows, the SwiGLU product of the two
//              feed-forward rows of a channel, or the residual addition
// Counterparts of Attention.forward, FeedForward.forward and RMSNorm of the reference's
// model (evaluation/dram-attention/model.py:66-78, :138-245) at sequence length 1.
//
// Bound: HBM, N*K*e bytes of weights read once (streaming loads: no step reads them twice).
// Every wave takes pairs of rows, so that what the endings need (a channel pair to rotate,
// the gate and up row of a channel) meets in one wave: 64 lanes x 16 bytes of each row per
// step, kUnroll steps of loads in flight per wave before the first is used; the input row
// is read from LDS, packed dot products into fp32, one fold over the wave per pair.
// Workgroups of four waves, no more than are resident at once (98 registers a wave: four
// workgroups per compute unit, fewer where the input row's LDS says so), every wave a pair in
// turn: all waves end within a pair of each other.  us, up to 2048 workgroups with consecutive pairs per
// wave (whose second round found half the chip idle) / this: output projection and
// feed-forward of 2048 x 7168 26.3 / 24.6, of 4096 x 14336 70.4 / 68.5; vocabulary 32000 x 2048 25.7 / 23.9,
// 50257 x 1024 26.4 / 23.7, 128256 x 4096 166.6 / 162.7.
//
// Measured (bf16, in a decode step, each with its endings; in brackets the library products
// alone): vocabulary 128256 x 4096 160 us = 6.6 TB/s (188); 2 x 14336 x 4096 39 us = 6.0 TB/s
// (57); 4096 x 14336 22 us (26); queries, keys and values 6144 x 4096 11.5 us (44 in three
// launches).  A token through four such layers over 32K-token prefixes, one graph, library products /
// these: 1.41 / 1.04 ms; through four layers of dim 2048 from Python, 72 / 38 launches: 1.38 / 0.67 ms.
#include "attention_core.hpp"
#include "model_math.hpp"

namespace da {

constexpr int kLinThreads = 256;
constexpr int kLinWaves = kLinThreads / 64;
constexpr int kLinUnroll = 4;
constexpr int kLinMaxRow = 60 * 1024;   // bytes of the input row (LDS)
constexpr int64_t kLinUnits = 256, kLinPerUnit = 4;  // compute units, resident workgroups of each
constexpr size_t kLinLds = 160 * 1024;

enum LinearEnd { kEndRope, kEndSwiglu, kEndAdd, kEndLogits };

struct LinearArgs {
  const char *x;
  const char *norm_weight;  // null: x as it is
  float eps;
  int dim;                  // K
  const char *w[3];         // rope: wq, wk, wv; swiglu: w1, w3; else w[0]
  int64_t n_pairs;
  // rope: rows of wq and of wk (and of wv), channels of a head, cosine and sine per pair
  int q_rows, kv_rows, head_dim;
  const float *rope;
  char *out[3];
  const char *residual;
  int64_t n_out;
};

template <typename T, int kEnd>
__global__ void __launch_bounds__(kLinThreads)
decode_linear_kernel(const LinearArgs a) {
  extern __shared__ __align__(16) char xs[];   // the input row, zeroes up to a whole step
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int vecs = a.dim / T::kVec;
  const int steps = (vecs + 63) / 64;
  const int64_t row_b = (int64_t)a.dim * T::kBytes;
  int64_t pair = (int64_t)blockIdx.x * kLinWaves + wave;
  const int64_t n_waves = (int64_t)gridDim.x * kLinWaves;

  // the two rows of a pair, and (rope) which matrix they belong to
  auto rows_of = [&](int64_t p, const char *&r0, const char *&r1) {
    if constexpr (kEnd == kEndSwiglu) {
      r0 = a.w[0] + p * row_b;
      r1 = a.w[1] + p * row_b;
    } else if constexpr (kEnd == kEndRope) {
      int64_t r = 2 * p;
      const char *base = a.w[0];
      if (r >= a.q_rows) {
        r -= a.q_rows;
        base = a.w[1];
        if (r >= a.kv_rows) {
          r -= a.kv_rows;
          base = a.w[2];
        }
      }
      r0 = base + r * row_b;
      r1 = r0 + row_b;
    } else {
      r0 = a.w[0] + 2 * p * row_b;
      r1 = 2 * p + 1 < a.n_out ? r0 + row_b : r0;   // an odd last row is read twice
    }
  };
  u32x4 w0[kLinUnroll], w1[kLinUnroll];
  auto load = [&](const char *r0, const char *r1, int s0) {
    if ((s0 + kLinUnroll) * 64 <= vecs) {
#pragma unroll
      for (int u = 0; u < kLinUnroll; ++u) {
        const int64_t at = ((int64_t)(s0 + u) * 64 + lane) * 16;
        w0[u] = load16_stream(r0 + at);
        w1[u] = load16_stream(r1 + at);
      }
    } else {
#pragma unroll
      for (int u = 0; u < kLinUnroll; ++u) {
        const int j = (s0 + u) * 64 + lane;
        w0[u] = w1[u] = u32x4{0, 0, 0, 0};
        if (j < vecs) {
          w0[u] = load16_stream(r0 + (int64_t)j * 16);
          w1[u] = load16_stream(r1 + (int64_t)j * 16);
        }
      }
    }
  };

  const char *r0, *r1;
  const bool any = pair < a.n_pairs;
  rows_of(any ? pair : a.n_pairs - 1, r0, r1);
  load(r0, r1, 0);

  // the input row into LDS
  {
    float inv = 0.f;
    if (a.norm_weight != nullptr) {
      float ss = 0.f;
      for (int j = threadIdx.x; j < vecs; j += kLinThreads) {
        float f[T::kVec];
        unpack<T>(load16(a.x + (int64_t)j * 16), f);
        ss += sum_of_squares<T>(f);
      }
      ss = group_sum<64>(ss);
      __shared__ float part[kLinWaves];
      if (lane == 0) part[wave] = ss;
      __syncthreads();
      static_assert(kLinWaves == 4, "the waves' sums in pairs");
      ss = (part[0] + part[1]) + (part[2] + part[3]);
      inv = rms_scale(ss, a.dim, a.eps);
    }
    const int padded = (steps + kLinUnroll - 1) / kLinUnroll * kLinUnroll * 64;
    for (int j = threadIdx.x; j < padded; j += kLinThreads) {
      u32x4 v = {0, 0, 0, 0};
      if (j < vecs) {
        v = load16(a.x + (int64_t)j * 16);
        if (a.norm_weight != nullptr) {
          float f[T::kVec], w[T::kVec];
          unpack<T>(v, f);
          unpack<T>(load16(a.norm_weight + (int64_t)j * 16), w);
#pragma unroll
          for (int i = 0; i < T::kVec; ++i) f[i] = round_to<T>(f[i] * inv) * w[i];
          v = pack_vec<T>(f);
        }
      }
      *(u32x4 *)(xs + j * 16) = v;
    }
  }
  __syncthreads();
  if (!any) return;

  float y0 = 0.f, y1 = 0.f;
  int s0 = 0;
  for (;;) {
#pragma unroll
    for (int u = 0; u < kLinUnroll; ++u) {
      const u32x4 xv = *(const u32x4 *)(xs + ((s0 + u) * 64 + lane) * 16);
      y0 += dot16<T>(xv, w0[u]);
      y1 += dot16<T>(xv, w1[u]);
    }
    s0 += kLinUnroll;
    const int64_t done = pair;
    if (s0 >= steps) {
      s0 = 0;
      pair += n_waves;
      if (pair < a.n_pairs) rows_of(pair, r0, r1);
    }
    const bool more = pair < a.n_pairs;
    if (more) load(r0, r1, s0);
    if (pair == done) continue;
    // a pair is complete
    y0 = round_to<T>(group_sum<64>(y0));
    y1 = round_to<T>(group_sum<64>(y1));
    if (lane == 0) {
      if constexpr (kEnd == kEndRope) {
        int64_t r = 2 * done;
        int which = 0;
        if (r >= a.q_rows) {
          r -= a.q_rows;
          which = 1;
          if (r >= a.kv_rows) {
            r -= a.kv_rows;
            which = 2;
          }
        }
        if (which < 2) {
          const float *cs = a.rope + r % a.head_dim;
          rotate_pair(y0, y1, cs[0], cs[1]);
        }
        store_elem<T>(a.out[which], r, y0);
        store_elem<T>(a.out[which], r + 1, y1);
      } else if constexpr (kEnd == kEndSwiglu) {
        store_elem<T>(a.out[0], done, round_to<T>(silu<T>(y0)) * y1);
      } else if constexpr (kEnd == kEndAdd) {
        store_elem<T>(a.out[0], 2 * done, load_elem<T>(a.residual, 2 * done) + y0);
        if (2 * done + 1 < a.n_out)
          store_elem<T>(a.out[0], 2 * done + 1, load_elem<T>(a.residual, 2 * done + 1) + y1);
      } else {
        store_elem<F32>(a.out[0], 2 * done, y0);
        if (2 * done + 1 < a.n_out) store_elem<F32>(a.out[0], 2 * done + 1, y1);
      }
    }
    if (!more) return;
    y0 = y1 = 0.f;
  }
}

// Index of the largest logit (the lowest of equal ones; a NaN counts as the largest, as in
// torch.argmax).  One workgroup: half a megabyte of logits, just written, comes from cache, without a
// second launch or a hand-over between workgroups.  Bound: the latency of its loads, 16 in
// flight per thread, once the arithmetic is short: a thread keeps the best of its vectors of four
// values, not of its values (a maximum and an index per vector), and whether there was a NaN at all; which
// value of the best vector it was is looked up at the end, and only a row with a NaN is gone
// through again.  128256 logits: 9.5 us (a key and an index per value 13.5, torch's reduction 40).
constexpr int kArgmaxThreads = 1024, kArgmaxLoads = 16;
__global__ void __launch_bounds__(kArgmaxThreads)
argmax_kernel(const float *__restrict__ x, int64_t n, int64_t *__restrict__ out) {
  constexpr uint32_t kNone = 0xffffffffu;
  __shared__ float part_best[kArgmaxThreads / 64];
  __shared__ uint32_t part_at[kArgmaxThreads / 64];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t vecs = n / 4;
  float best = -INFINITY;
  uint32_t at = kNone;        // vector of the best value, the lowest (n < 2^31)
  bool nan = false;
  for (int64_t j0 = t; j0 < vecs; j0 += kArgmaxLoads * kArgmaxThreads) {
    float4 v[kArgmaxLoads];
#pragma unroll
    for (int u = 0; u < kArgmaxLoads; ++u) {
      const int64_t j = j0 + u * kArgmaxThreads;
      v[u] = *(const float4 *)(x + 4 * (j < vecs ? j : j0));
    }
#pragma unroll
    for (int u = 0; u < kArgmaxLoads; ++u) {
      const int64_t j = j0 + u * kArgmaxThreads;
      nan |= __builtin_isunordered(v[u].x, v[u].y) || __builtin_isunordered(v[u].z, v[u].w);
      const float m = fmaxf(fmaxf(v[u].x, v[u].y), fmaxf(v[u].z, v[u].w));
      if (j < vecs && (m > best || at == kNone)) {     // (a row of -inf has a best too)
        best = m;
        at = (uint32_t)j;
      }
    }
  }
  // the last n % 4 values as a vector of their own
  if (t == 0)
    for (int64_t i = 4 * vecs; i < n; ++i) {
      nan |= x[i] != x[i];
      if (x[i] > best || at == kNone) {
        best = x[i];
        at = (uint32_t)vecs;
      }
    }
  if (__syncthreads_or(nan)) {
    uint32_t first = kNone;
    for (int64_t i = t; i < n; i += kArgmaxThreads)
      if (x[i] != x[i]) {
        first = (uint32_t)i;
        break;
      }
    for (int m = 32; m >= 1; m >>= 1) first = min(first, (uint32_t)__shfl_xor((int)first, m, 64));
    if (lane == 0) part_at[wave] = first;
    __syncthreads();
    if (t == 0) {
      for (int i = 1; i < kArgmaxThreads / 64; ++i) first = min(first, part_at[i]);
      *out = (int64_t)first;
    }
    return;
  }
  // (a thread without a vector: -inf at kNone, behind every other)
  auto better = [](float b, uint32_t i, float c, uint32_t k) { return c > b || (c == b && k < i); };
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    const float c = __shfl_xor(best, m, 64);
    const uint32_t k = (uint32_t)__shfl_xor((int)at, m, 64);
    if (better(best, at, c, k)) {
      best = c;
      at = k;
    }
  }
  if (lane == 0) {
    part_best[wave] = best;
    part_at[wave] = at;
  }
  __syncthreads();
  if (t == 0) {
    for (int i = 1; i < kArgmaxThreads / 64; ++i)
      if (better(best, at, part_best[i], part_at[i])) {
        best = part_best[i];
        at = part_at[i];
      }
    int64_t i = 4 * (int64_t)at;
    while (x[i] != best) ++i;      // (no NaN: the vector, or the rest of the row, holds it)
    *out = i;
  }
}

template <int kEnd>
static int launch_linear(const char *what, LinearArgs a, int dtype, hipStream_t s) {
  DA_REQUIRE(dtype == DA_F32 || dtype == DA_F16 || dtype == DA_BF16, "%s: unknown dtype %d", what, dtype);
  DA_REQUIRE(a.dim > 0 && a.n_out > 0, "%s: bad shape", what);
  DA_REQUIRE(a.x && a.w[0] && a.out[0], "%s: null pointer", what);
  const int64_t row_b = (int64_t)a.dim * elem_size(dtype);
  if (row_b % 16 != 0 || row_b > kLinMaxRow)
    return fail(DA_ENOTSUP, "%s: input rows of a multiple of 16 bytes up to 60 KiB (got %lld)", what,
                (long long)row_b);
  for (const void *p : {(const void *)a.x, (const void *)a.norm_weight, (const void *)a.w[0],
                        (const void *)a.w[1], (const void *)a.w[2]})
    DA_REQUIRE((uintptr_t)p % 16 == 0, "%s: operands must be 16-byte aligned", what);
  const size_t lds = (size_t)ceil_div(row_b, 1024 * kLinUnroll) * 1024 * kLinUnroll;
  const int64_t fit = (int64_t)(kLinLds / (lds + 64)), most = kLinUnits * (fit < kLinPerUnit ? fit : kLinPerUnit);
  const int64_t wanted = ceil_div(a.n_pairs, (int64_t)kLinWaves);
  const int64_t blocks = wanted < most ? wanted : most;
  const dim3 grid((unsigned)blocks);
#define DA_LINEAR(T) hipLaunchKernelGGL((decode_linear_kernel<T, kEnd>), grid, dim3(kLinThreads), lds, s, a)
  if (dtype == DA_BF16) DA_LINEAR(BF16);
  else if (dtype == DA_F16) DA_LINEAR(F16);
  else DA_LINEAR(F32);
#undef DA_LINEAR
  return launch_status(what);
}

}  // namespace da

extern "C" int da_linear_qkv_rope(const void *x, const void *norm_weight, float eps, int dim, const void *wq,
                                  const void *wk, const void *wv, int n_q_heads, int n_kv_heads, int head_dim,
                                  const float *rope_row, void *q_out, void *k_out, void *v_out, int dtype,
                                  void *stream) {
  using namespace da;
  DA_REQUIRE(n_q_heads > 0 && n_kv_heads > 0 && head_dim > 0 && head_dim % 2 == 0,
             "da_linear_qkv_rope: bad heads");
  DA_REQUIRE(wk && wv && rope_row && k_out && v_out, "da_linear_qkv_rope: null pointer");
  if ((int64_t)n_q_heads * head_dim > 0x3fffffff || (int64_t)n_kv_heads * head_dim > 0x3fffffff)
    return fail(DA_ENOTSUP, "da_linear_qkv_rope: too many rows");
  LinearArgs a = {};
  a.x = (const char *)x;
  a.norm_weight = (const char *)norm_weight;
  a.eps = eps;
  a.dim = dim;
  a.w[0] = (const char *)wq;
  a.w[1] = (const char *)wk;
  a.w[2] = (const char *)wv;
  a.q_rows = n_q_heads * head_dim;
  a.kv_rows = n_kv_heads * head_dim;
  a.head_dim = head_dim;
  a.rope = rope_row;
  a.out[0] = (char *)q_out;
  a.out[1] = (char *)k_out;
  a.out[2] = (char *)v_out;
  a.n_out = (int64_t)a.q_rows + 2 * a.kv_rows;
  a.n_pairs = a.n_out / 2;
  return launch_linear<kEndRope>("da_linear_qkv_rope", a, dtype, (hipStream_t)stream);
}

extern "C" int da_linear_swiglu(const void *x, const void *norm_weight, float eps, int dim, const void *w1,
                                const void *w3, int64_t hidden, void *out, int dtype, void *stream) {
  using namespace da;
  DA_REQUIRE(w3, "da_linear_swiglu: null pointer");
  LinearArgs a = {};
  a.x = (const char *)x;
  a.norm_weight = (const char *)norm_weight;
  a.eps = eps;
  a.dim = dim;
  a.w[0] = (const char *)w1;
  a.w[1] = (const char *)w3;
  a.out[0] = (char *)out;
  a.n_out = a.n_pairs = hidden;
  return launch_linear<kEndSwiglu>("da_linear_swiglu", a, dtype, (hipStream_t)stream);
}

extern "C" int da_linear_add(const void *x, int dim, const void *w, int64_t n_out, const void *residual, void *out,
                             int dtype, void *stream) {
  using namespace da;
  DA_REQUIRE(residual, "da_linear_add: null pointer");
  LinearArgs a = {};
  a.x = (const char *)x;
  a.dim = dim;
  a.w[0] = (const char *)w;
  a.out[0] = (char *)out;
  a.residual = (const char *)residual;
  a.n_out = n_out;
  a.n_pairs = ceil_div(n_out, 2);
  return launch_linear<kEndAdd>("da_linear_add", a, dtype, (hipStream_t)stream);
}

extern "C" int da_linear_logits(const void *x, const void *norm_weight, float eps, int dim, const void *w,
                                int64_t n_out, float *out, int dtype, void *stream) {
  using namespace da;
  LinearArgs a = {};
  a.x = (const char *)x;
  a.norm_weight = (const char *)norm_weight;
  a.eps = eps;
  a.dim = dim;
  a.w[0] = (const char *)w;
  a.out[0] = (char *)out;
  a.n_out = n_out;
  a.n_pairs = ceil_div(n_out, 2);
  return launch_linear<kEndLogits>("da_linear_logits", a, dtype, (hipStream_t)stream);
}

extern "C" int da_linear_block_tail(const void *attn, int attn_dim, const void *wo, const void *x, int dim,
                                    const void *norm_weight, float eps, const void *w1, const void *w3,
                                    int hidden, const void *w2, void *h, void *act, void *out, int dtype,
                                    void *stream) {
  int rc = da_linear_add(attn, attn_dim, wo, dim, x, h, dtype, stream);
  if (rc) return rc;
  rc = da_linear_swiglu(h, norm_weight, eps, dim, w1, w3, hidden, act, dtype, stream);
  if (rc) return rc;
  return da_linear_add(act, hidden, w2, dim, h, out, dtype, stream);
}

extern "C" int da_argmax(const float *x, int64_t n, int64_t *out, void *stream) {
  using namespace da;
  DA_REQUIRE(n > 0 && n <= 0x7fffffff, "da_argmax: 1 to 2^31 - 1 values");
  DA_REQUIRE(x && out && (uintptr_t)x % 16 == 0, "da_argmax: null or unaligned pointer");
  hipLaunchKernelGGL(argmax_kernel, dim3(1), dim3(kArgmaxThreads), 0, (hipStream_t)stream, x, n, out);
  return launch_status("da_argmax");
}
