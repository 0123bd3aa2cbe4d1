// Causal attention over the whole prompt in fp32: the form of prefill_attention.hip
// for float keys, values and queries, on the fp32 matrix instructions (every product
// and sum in fp32).  Counterpart of flash_attn_func(xq, xk, xv, causal=True) in
// dram_attention/dram_attention.py:136 of the reference for an fp32 layer.
//
// Bound: fp32 MFMA (64 flops per cycle and SIMD, a sixteenth of the bf16 rate), so what
// counts is that the matrix cores of all SIMDs stay busy to the end; LDS (a quarter of its
// rate) and the softmax (an eighth of the MFMA time) hide behind them.
//
// Work split: a 256-thread workgroup owns kHeads query heads of one kv head times
// 64/kHeads consecutive query rows; each of its four waves owns 16 rows of one head.
// 16-row waves (v_mfma_f32_16x16x4_f32) and not 32-row ones: the rate is the same, and the
// longest row block, which nothing shortens, is half as long.  Per tile of 32 keys in LDS:
//   S^T (keys x rows)  = K (keys x D) * Q^T (D x rows)       D/4 MFMAs per 16 keys
//   O^T (D x rows)    += V^T (D x keys) * P^T (keys x rows)  D/16 MFMAs per 4 keys
// Lane (g, c) = (l / 16, l % 16) gets row c, keys 4g + i of S^T in register i, which is,
// register by register, the B operand of the second product (k index g is key 4g + i): the
// weights go from one product to the other without a move.  Both contractions may run in
// any order and output channels may sit anywhere, so the channels are dealt out to suit
// 16-byte LDS reads: a lane's four consecutive channels 16t + 4g .. +3 of a K row are its A
// operands of four steps, and its four consecutive channels 4c .. +3 of a V row its A
// operands of four channel blocks (block b, row c is channel 4c + b).
//
// Measured: 133 TFLOP/s (0.85 of 157; a large fp32 matrix product of the library: 154) at 32/8
// heads, D 128, 9200 tokens; 0.70 ms = 125 TFLOP/s at 8/2 heads, D 64, 9200 tokens, where
// torch's operators took 4.27 ms.
//
// Sums: a score is the sum of two chains of MFMAs, over every other 16 channels each, and a lane
// adds its eight weights of a tile in pairs before they join its running sum.  Distance to
// float64 (2-norm; N(0, 1) queries and values, keys with outlier channels) in single chains / like
// this / of torch's blocked operators, in 1e-7: 8/2 heads, D 64: 1756 tokens 5.1 / 4.2 / 4.7, 3000 5.9
// / 5.0 / 5.5, 9200 8.5 / 7.6 / 8.4; 16/4 2500: 5.5 / 4.7 / 5.3; 32/8, D 128: 1800 5.9 / 4.5 / 5.9, 9000 8.5 /
// 7.4 / 8.5.  It costs 1 % at 9200 tokens of 8/2 heads (688 -> 695 us) and nothing at D 128.  (Output
// sums of 16 tiles joining a second set of registers: 4.6, 4.9, 5.4, but the kernel then fills the
// register file, and the page store beside it takes 5 % more of the call.)
//
// Tiles are double-buffered and travel global memory -> LDS directly, in the blocks of
// 1024 bytes with swizzled columns that prefill_attention.hip explains.
#include <type_traits>

#include "prefill_args.hpp"

namespace da {

typedef float pf_f32x4 __attribute__((ext_vector_type(4)));

constexpr int kPfsThreads = 256;
constexpr int kPfsWaves = 4;
constexpr int kPfsRows = 16;  // query rows of a wave
constexpr int kPfsKeys = 32;  // keys per tile
constexpr int kPfsCus = 256;      // compute units of the part
constexpr int kPfsResident = 4;   // workgroups of one launch a unit holds at once (two at D 128)

template <int kD>
struct PrefillSharedF32 {
  static constexpr int kRowBytes = kD * 4;
  static constexpr int kRows = 1024 / kRowBytes;   // rows per block: 4 (D 64) or 2 (D 128)
  static constexpr int kChunks = kRowBytes / 16;   // 16-byte chunks per row
  static constexpr int kBlock = 1024 + 16;         // bytes from block to block
  static constexpr int kBlocks = kPfsKeys / kRows; // blocks per tile (K, and V)
  static constexpr int kKBytes = kBlocks * kBlock;
  static constexpr int kBufBytes = 2 * kKBytes;    // K tile, then V tile
  // 16 lanes that read one column of 16 rows (K operands) fall on 16 different columns
  // modulo 16: kRows rows by the swizzle, the blocks by their padding
  static __host__ __device__ constexpr int swizzle(int rr) { return (16 / kRows) * rr; }
  static __device__ __forceinline__ int at(int r, int cc) {
    return (r / kRows) * kBlock + (r % kRows) * kRowBytes + ((cc ^ swizzle(r % kRows)) * 16);
  }
};

template <int kD, int kHeads>
__global__ void __launch_bounds__(kPfsThreads, 2)
prefill_attention_f32_kernel(const PrefillArgs a, const int n_kv_heads) {
  using Sh = PrefillSharedF32<kD>;
  if (prefill_gate(a)) return;
  static_assert(kD == 64 || kD == 128, "head sizes of 64 and 128");
  constexpr int kBlockRows = kPfsRows * kPfsWaves / kHeads;
  constexpr int kQChunks = kD / 16;     // 16-byte query chunks per lane
  constexpr int kCGroups = kD / 64;     // groups of 64 output channels
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int g = lane >> 4;
  const int c = lane & 15;

  // Longest rows first over all heads.  The first kPfsResident workgroups per compute unit
  // start together, number j of each 256 on the same unit, and then share its matrix cores:
  // every other 256 of them is turned round, so that a unit with a longest block gets a short
  // one with it (9200 tokens, 8/2 heads: 0.747 against 0.836 ms; 3000 tokens, 16/16: 0.187
  // against 0.211).  Later workgroups go wherever one ends.
  unsigned b = blockIdx.x;
  if (b / kPfsCus % 2 == 1 && b < kPfsResident * kPfsCus && (b / kPfsCus + 1) * kPfsCus <= gridDim.x)
    b = (b / kPfsCus + 1) * kPfsCus - 1 - b % kPfsCus;
  const int hk = (int)(b % (unsigned)n_kv_heads);
  const int64_t rem = b / (unsigned)n_kv_heads;
  const int64_t rb = a.n_row_blocks - 1 - rem / a.n_groups;
  const int hq = hk * a.rep + (int)(rem % a.n_groups) * kHeads + wave % kHeads;
  const int64_t S = a.seq_len;
  const int64_t m0 = rb * kBlockRows;
  const int64_t row0 = m0 + (wave / kHeads) * kPfsRows;
  const int64_t my_row = row0 + c;
  const int64_t last_key = (m0 + kBlockRows < S ? m0 + kBlockRows : S) - 1;
  const int n_tiles = (int)(last_key / kPfsKeys) + 1;
  const int64_t wave_last_key = row0 + kPfsRows - 1 < S ? row0 + kPfsRows - 1 : S - 1;

  __shared__ __align__(16) char smem[2 * Sh::kBufBytes];

  // Q^T as the B operand: row c, channels 16t + 4g .. +3
  u32x4 qf[kQChunks];
  {
    const int64_t r = my_row < S ? my_row : S - 1;
    const char *qp = a.q + (r * a.q_tok_stride + (int64_t)hq * a.q_head_stride) * 4 + g * 16;
#pragma unroll
    for (int t = 0; t < kQChunks; ++t) qf[t] = load16(qp + t * 64);
  }

  const char *kbase = a.k + (int64_t)hk * a.k_head_stride * 4;
  const char *vbase = a.v + (int64_t)hk * a.v_head_stride * 4;
  const int64_t k_tok_b = a.k_tok_stride * 4, v_tok_b = a.v_tok_stride * 4;

  constexpr int kBlocksPerWave = Sh::kBlocks / kPfsWaves;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int ld_row = lane / Sh::kChunks;
  const int ld_col = (lane % Sh::kChunks) ^ Sh::swizzle(ld_row);
  typedef __attribute__((address_space(1))) const void *GlobalPtr;
  typedef __attribute__((address_space(3))) void *LdsPtr;
  const uint32_t k_rel = (uint32_t)(ld_row * k_tok_b) + ld_col * 16;   // (fit 32 bits: checked by the launcher)
  const uint32_t v_rel = (uint32_t)(ld_row * v_tok_b) + ld_col * 16;
  auto fetch = [&](int tile, int buf) {
    const int64_t t0 = (int64_t)tile * kPfsKeys;
    char *kt = smem + buf * Sh::kBufBytes;
    if (t0 + kPfsKeys - 1 <= last_key) {            // a whole tile: one base, constant offsets
      const char *kt0 = kbase + t0 * k_tok_b, *vt0 = vbase + t0 * v_tok_b;
#pragma unroll
      for (int u = 0; u < kBlocksPerWave; ++u) {
        const int blk = wave_u + u * kPfsWaves;
        __builtin_amdgcn_global_load_lds((GlobalPtr)(kt0 + (int64_t)blk * Sh::kRows * k_tok_b + k_rel),
                                         (LdsPtr)(kt + blk * Sh::kBlock), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((GlobalPtr)(vt0 + (int64_t)blk * Sh::kRows * v_tok_b + v_rel),
                                         (LdsPtr)(kt + Sh::kKBytes + blk * Sh::kBlock), 16, 0, 0);
      }
    } else {
#pragma unroll
      for (int u = 0; u < kBlocksPerWave; ++u) {
        const int blk = wave_u + u * kPfsWaves;
        int64_t tok = t0 + blk * Sh::kRows + ld_row;
        if (tok > last_key) tok = last_key;         // in bounds; such keys are masked
        __builtin_amdgcn_global_load_lds((GlobalPtr)(kbase + tok * k_tok_b + ld_col * 16),
                                         (LdsPtr)(kt + blk * Sh::kBlock), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((GlobalPtr)(vbase + tok * v_tok_b + ld_col * 16),
                                         (LdsPtr)(kt + Sh::kKBytes + blk * Sh::kBlock), 16, 0, 0);
      }
    }
  };

  // LDS places of this lane's operands: K row c of a 16-key half, chunk 4t + g; V row
  // 4g + i of a half, chunk c (of each 64 channels).
  int k_at[kQChunks], v_at[4][kCGroups];
#pragma unroll
  for (int t = 0; t < kQChunks; ++t) k_at[t] = Sh::at(c, 4 * t + g);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int q = 0; q < kCGroups; ++q) v_at[i][q] = Sh::kKBytes + Sh::at(4 * g + i, 16 * q + c);
  constexpr int kHalfStep = (16 / Sh::kRows) * Sh::kBlock;

  float m = kMinusHuge, l = 0.f;
  pf_f32x4 acc[4 * kCGroups];   // [4q + b]: rows 4g + i are channels 64q + 16g + 4i + b
#pragma unroll
  for (int b = 0; b < 4 * kCGroups; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[b][i] = 0.f;

  auto compute = [&](int tile, int buf, auto mask_tag) {
    constexpr bool kMask = decltype(mask_tag)::value;
    __builtin_amdgcn_iglp_opt(1);   // (measured: see the loop below)
    const char *kt = smem + buf * Sh::kBufBytes;
    pf_f32x4 st[2], odd[2];   // the channels' sums in two chains (chunks of 16 in turn)
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < 4; ++i) st[half][i] = odd[half][i] = 0.f;
#pragma unroll
    for (int t = 0; t < kQChunks; t += 2) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const u32x4 k0 = *(const u32x4 *)(kt + k_at[t + u]);
        const u32x4 k1 = *(const u32x4 *)(kt + k_at[t + u] + kHalfStep);
        pf_f32x4 *const s = u ? odd : st;
#pragma unroll
        for (int i = 0; i < 4; ++i) {   // the two halves in turn: each chain's latency hides the other's
          s[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(as_f32(k0[i]), as_f32(qf[t + u][i]), s[0], 0, 0, 0);
          s[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(as_f32(k1[i]), as_f32(qf[t + u][i]), s[1], 0, 0, 0);
        }
      }
    }
    st[0] += odd[0];
    st[1] += odd[1];
    float smax = -INFINITY;
    if constexpr (kMask) {
      const int lim = (int)(my_row - ((int64_t)tile * kPfsKeys + 4 * g));  // key offset <= lim stays
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (half * 16 + i > lim) st[half][i] = -INFINITY;
    }
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < 4; ++i) smax = fmaxf(smax, st[half][i]);
    smax *= a.scale_log2;   // the scale is positive: max and scaling commute
    if (__any(smax > m + kRescaleSlack)) {  // rare after the first tiles
      float mx = fmaxf(m, smax);
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float alpha = fast_exp2(m - mx);
      m = mx;
      l *= alpha;
#pragma unroll
      for (int b = 0; b < 4 * kCGroups; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[b][i] *= alpha;
    }
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < 4; ++i) st[half][i] = fast_exp2(fmaf(st[half][i], a.scale_log2, -m));
    l += ((st[0][0] + st[0][1]) + (st[0][2] + st[0][3])) + ((st[1][0] + st[1][1]) + (st[1][2] + st[1][3]));
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < kCGroups; ++q) {
          const u32x4 va = *(const u32x4 *)(kt + v_at[i][q] + half * kHalfStep);
#pragma unroll
          for (int b = 0; b < 4; ++b)
            acc[4 * q + b] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(as_f32(va[b]), st[half][i], acc[4 * q + b], 0, 0, 0);
        }
  };

  fetch(0, 0);
#pragma unroll
  for (int t = 0; t < kQChunks; ++t) asm volatile("" : "+v"(qf[t]));  // (arrived before the loop)
  __syncthreads();
  // Tiles below the workgroup's first row, which every wave needs whole, go two a round, as
  // in prefill_attention.hip: with the buffer known at compile time LDS addresses are a
  // register plus a constant, and a whole tile's loads one base plus constants (a 64-bit
  // product per lane and load before).  iglp_opt(1) spreads the LDS reads between the MFMAs.
  // us as it was / with the rounds / and iglp_opt (same bits): 9200 tokens, 8/2 heads, D 64: 743 /
  // 696 / 687; 1800: 82.9 / 75.6 / 72.9; 9000, 16/4: 1381 / 1298 / 1281; 9200, 32/8, D 128: 5518 / 5325 / 5222.
  const int n_whole = (int)(m0 / kPfsKeys) & ~1;
  for (int tile = 0; tile < n_whole; tile += 2) {
    fetch(tile + 1, 1);
    compute(tile, 0, std::false_type{});
    __syncthreads();
    fetch(tile + 2, 0);                             // (there is one: the tiles of the block's own rows)
    compute(tile + 1, 1, std::false_type{});
    __syncthreads();
  }
  for (int tile = n_whole; tile < n_tiles; ++tile) {
    const int buf = tile & 1;
    if (tile + 1 < n_tiles) fetch(tile + 1, buf ^ 1);
    const int64_t t0 = (int64_t)tile * kPfsKeys;
    if (t0 <= wave_last_key) {
      if (t0 + kPfsKeys - 1 > row0) compute(tile, buf, std::true_type{});
      else compute(tile, buf, std::false_type{});
    }
    __syncthreads();
  }

  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  if (my_row < S) {
    float *op = (float *)(a.out + (my_row * a.o_tok_stride + (int64_t)hq * a.o_head_stride) * 4) + 16 * g;
#pragma unroll
    for (int q = 0; q < kCGroups; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const pf_f32x4 o = {acc[4 * q][i] * inv, acc[4 * q + 1][i] * inv, acc[4 * q + 2][i] * inv,
                            acc[4 * q + 3][i] * inv};
        *(pf_f32x4 *)(op + 64 * q + 4 * i) = o;
      }
    if (a.lse != nullptr && g == 0)
      a.lse[(int64_t)hq * S + my_row] = l > 0.f ? (m + __builtin_amdgcn_logf(l)) * kLn2 : -INFINITY;
  }
}

template <int kD>
static int launch_prefill_f32_of(PrefillArgs a, int n_kv_heads, hipStream_t s) {
  const int heads = a.rep % 4 == 0 ? 4 : (a.rep % 2 == 0 ? 2 : 1);
  a.n_groups = a.rep / heads;
  a.n_row_blocks = ceil_div(a.seq_len, kPfsRows * kPfsWaves / heads);
  const int64_t blocks = a.n_row_blocks * a.n_groups * n_kv_heads;
  if (blocks > 0x7fffffff)
    return fail(DA_ENOTSUP, "da_prefill_attention_f32: %lld workgroups", (long long)blocks);
  const dim3 grid((unsigned)blocks);
  if (heads == 4)
    hipLaunchKernelGGL((prefill_attention_f32_kernel<kD, 4>), grid, dim3(kPfsThreads), 0, s, a, n_kv_heads);
  else if (heads == 2)
    hipLaunchKernelGGL((prefill_attention_f32_kernel<kD, 2>), grid, dim3(kPfsThreads), 0, s, a, n_kv_heads);
  else
    hipLaunchKernelGGL((prefill_attention_f32_kernel<kD, 1>), grid, dim3(kPfsThreads), 0, s, a, n_kv_heads);
  return launch_status("da_prefill_attention_f32");
}

int launch_prefill_f32(const PrefillArgs &a, int head_dim, hipStream_t s) {
  return head_dim == 128 ? launch_prefill_f32_of<128>(a, a.n_kv_heads, s)
                         : launch_prefill_f32_of<64>(a, a.n_kv_heads, s);
}

}  // namespace da

extern "C" int da_prefill_attention_f32(const float *q, int64_t q_tok_stride, int64_t q_head_stride,
                                        const float *k, int64_t k_tok_stride, int64_t k_head_stride,
                                        const float *v, int64_t v_tok_stride, int64_t v_head_stride,
                                        int64_t seq_len, int n_q_heads, int n_kv_heads, int head_dim,
                                        float scale, float *out, int64_t o_tok_stride,
                                        int64_t o_head_stride, float *lse_out, void *stream) {
  using namespace da;
  PrefillArgs a = {};
  const int rc = prefill_args(a, "da_prefill_attention_f32", q, q_tok_stride, q_head_stride, k, k_tok_stride,
                              k_head_stride, v, v_tok_stride, v_head_stride, seq_len, n_q_heads, n_kv_heads,
                              DA_F32, scale, out, o_tok_stride, o_head_stride, lse_out);
  if (rc != DA_OK || seq_len == 0) return rc;
  if (head_dim != 64 && head_dim != 128)
    return fail(DA_ENOTSUP, "da_prefill_attention_f32: head_dim 64 or 128 (got %d)", head_dim);
  return launch_prefill_f32(a, head_dim, (hipStream_t)stream);
}
