// Causal attention over a longer fp32 prompt on the bf16 matrix instructions, at fp32
// precision: every operand is held as the sum of three bf16 numbers.  The same result as
// prefill_attention_f32.hip, counterpart of flash_attn_func(xq, xk, xv, causal=True) in
// dram_attention/dram_attention.py:136 of the reference for an fp32 layer.
//
// Arithmetic.  a = a1 + a2 + a3 with a1 = bf16(a), a2 = bf16(a - a1), a3 = bf16(a - a1 - a2):
// both differences are exact and 3 x 8 bits and two signs cover the 24 of a float, so the
// sum IS a.  Of the nine products of two such operands six are formed, a1b1, a1b2, a2b1, a2b2,
// a1b3, a3b1; each is exact in fp32, and the three left out are at most 2^-26 of the whole, a
// quarter of the rounding of one fp32 addition.  The five small products have an accumulator of
// their own, so a score's large products meet in D/16 additions (of 16 products each) instead
// of D/4, and an output's in one for every 16 keys instead of every 4.  Queries, keys, values
// and softmax weights are split alike; softmax, its sums and the outputs are fp32.
//
// Weights reach down to 2^-126, where second and third parts would fall below the normal numbers (a
// weight of 2^-121 kept to 2.6e-4), so they are split as 2^24 times themselves: the smallest
// third part is then a normal number, and the sums of 2^31 weights of 2^8 and values of 2^60 end at 2^123.
// Exact, and taken back with the division by the sum; us without / with it: 9200 tokens, 8/2 heads,
// D 64: 457 / 466; 9000, 32/8, D 128: 3196 / 3217.
//
// Operands for which that is not so (not finite, above 2^60 or, but for zero, below 2^-100:
// infinite products, third parts that fp32's own range cuts off) are looked for by the kernel
// that splits keys and values, which leaves a word per workgroup; if one is set, this file's
// attention kernel does nothing and the one of prefill_attention_f32.hip, launched behind
// it and returning at once otherwise, does the prompt.
//
// Distance to float64 (2-norm; N(0, 1) queries and values, keys with outlier channels) of the plain
// kernel / of this one, in 1e-7: 8/2 heads, D 64: 300 tokens 2.4 / 1.4, 1756 4.2 / 2.0, 9200 7.6 / 2.8; 16/16,
// 5000: 6.0 / 2.3; 32/8, D 128: 700 3.5 / 1.8, 9000 7.4 / 2.4.
//
// Bound: MFMA, six bf16 products at 1024 flops per cycle and SIMD: 171 against the 64 of the
// fp32 instructions.  us of the plain kernel / of the three launches here: 9200 tokens, 8/2 heads,
// D 64: 695 / 466 (1.12 PFLOP/s of bf16 products; a large bf16 matrix product of the library: 1.36);
// 5000, 16/16, D 64: 447 / 302; 9000, 32/8, D 128: 5006 / 3217 (1.24 PFLOP/s); 64/8, 2000, D 128: 532 / 367.
//
// Work split.  prefill_split_kernel writes keys and values once, split and in the order in which
// the matrix instructions take them: an operand of one instruction, 32 rows x 16 k indices
// of one part, is 1024 consecutive bytes, lane after lane.  Tiles then travel global memory ->
// LDS as straight copies, an operand is one conflict-free 16-byte LDS read per lane, and V
// needs no transposing.  A round is 64 keys: D/16 operands x 3 parts x 2 halves of K, as many
// of V, 48 KiB at D 64 and 96 KiB at D 128.  A 512-thread workgroup, one per compute unit, owns
// kHeads query heads of one kv head x 128/kHeads rows: four waves hold 32 rows of one head each
// and take the first 32 keys of every round, four more the same rows and the other 32 keys
// (two waves on every SIMD, one's softmax beside the other's products, and serial chains
// half as long as with 256 rows); their states meet at the end, in fp32 through LDS.
//
// The products are those of prefill_attention.hip (S^T = K Q^T, whose registers are the B operand
// of O^T += V^T P^T), with its order of keys inside an operand of V.
#include <type_traits>

#include "prefill_args.hpp"

namespace da {

typedef float ps_f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 ps_bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kPsThreads = 512;
constexpr int kPsKeys = 64;            // keys of a round, 32 for each group of waves
constexpr int kPsOperand = 1024;       // bytes of one operand of an MFMA
constexpr int kPsSplitThreads = 256;
constexpr float kWeightScale = 0x1p24f;  // of the softmax weights while they are split (see above)
constexpr int kPsMaxSplitBlocks = 1024;  // workgroups of the splitting kernel, a flag word each

template <int kD>
struct SplitShape {
  static constexpr int kSteps = kD / 16;                      // K operands of 32 keys, per part
  static constexpr int kHalf = kSteps * 3 * kPsOperand;       // K, or V, of 32 keys
  static constexpr int kSide = 2 * kHalf;                     // K, or V, of a round
  static constexpr int kRound = 2 * kSide;
  // LDS: K of two rounds; V of two rounds at D 64, of one at D 128 (160 KiB hold no more)
  static constexpr int kVBufs = kD == 64 ? 2 : 1;
  static constexpr int kTiles = (2 + kVBufs) * kSide;
  static constexpr int kStash = 4 * (kD / 8 + 1) * 1024;      // the second group's state, at the end
  static constexpr int kBytes = kTiles > kStash ? kTiles : kStash;
};

__device__ __forceinline__ ps_f32x16 ps_mma(const u32x4 &a, const u32x4 &b, const ps_f32x16 &c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(ps_bf16x8, a),
                                                 __builtin_bit_cast(ps_bf16x8, b), c, 0, 0, 0);
}

// (lo, hi) as three packed pairs of bf16.  x - bf16(x) by a dot product whose other half is
// zero: one instruction instead of an unpacking and a subtraction, and as exact.
__device__ __forceinline__ void split_pair(float lo, float hi, uint32_t &w1, uint32_t &w2, uint32_t &w3) {
  // (in registers of their own: (-1, 0) as a literal comes out of this compiler as the inline
  // constant -1.0f, which the instruction takes for (0, -1))
  uint32_t only_lo = 0x0000bf80u, only_hi = 0xbf800000u;
  asm("" : "+s"(only_lo), "+s"(only_hi));
  const bf16x2 minus_lo = as_bf16x2(only_lo), minus_hi = as_bf16x2(only_hi);
  w1 = pack_bf16(lo, hi);
  lo = __builtin_amdgcn_fdot2_f32_bf16(as_bf16x2(w1), minus_lo, lo, false);
  hi = __builtin_amdgcn_fdot2_f32_bf16(as_bf16x2(w1), minus_hi, hi, false);
  w2 = pack_bf16(lo, hi);
  lo = __builtin_amdgcn_fdot2_f32_bf16(as_bf16x2(w2), minus_lo, lo, false);
  hi = __builtin_amdgcn_fdot2_f32_bf16(as_bf16x2(w2), minus_hi, hi, false);
  w3 = pack_bf16(lo, hi);
}
__device__ __forceinline__ void split8(const float *f, u32x4 *part) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t w1, w2, w3;
    split_pair(f[2 * i], f[2 * i + 1], w1, w2, w3);
    part[0][i] = w1;
    part[1][i] = w2;
    part[2][i] = w3;
  }
}

// Whether the three parts of x, and their products, stand for x.
__device__ __forceinline__ bool splits(float x) {
  const float a = __builtin_fabsf(x);
  return a == 0.f || (a >= 0x1p-100f && a <= 0x1p60f);   // (false for NaN)
}

// Keys and values into operands, and a look at all three inputs.  Bound: memory, 4 bytes read
// and 6 written per element of K and V, 4 read per element of Q.  A wave writes the three parts
// of one operand at a time.
template <int kD>
__global__ void __launch_bounds__(kPsSplitThreads)
prefill_split_kernel(const PrefillArgs a, char *__restrict__ planes, uint32_t *__restrict__ flags,
                     const int64_t n_rounds) {
  using Sh = SplitShape<kD>;
  constexpr int kOps = 4 * Sh::kSteps;     // operands of a round, per part
  const int lane = threadIdx.x & 63;
  const int g = lane >> 5, c = lane & 31;
  const int64_t S = a.seq_len;
  bool bad = false;
  const int64_t n_items = n_rounds * kOps * a.n_kv_heads;
  const int64_t first = ((int64_t)blockIdx.x * kPsSplitThreads + threadIdx.x) >> 6;
  const int64_t stride = (int64_t)gridDim.x * (kPsSplitThreads / 64);
  for (int64_t item = first; item < n_items; item += stride) {
    const int op = (int)(item % kOps);
    const int64_t at = item / kOps;        // round of head: head * n_rounds + round
    const int64_t h = at / n_rounds, key0 = (at % n_rounds) * kPsKeys;
    char *dst = planes + at * Sh::kRound + lane * 16;
    float f[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = 0.f;  // keys past the prompt
    if (op < 2 * Sh::kSteps) {               // K: key c of a half, channels 16s + 8g .. +7
      const int half = op / Sh::kSteps, s = op % Sh::kSteps;
      const int64_t key = key0 + half * 32 + c;
      if (key < S) {
        const char *src = a.k + (key * a.k_tok_stride + h * a.k_head_stride + s * 16 + g * 8) * 4;
        const u32x4 lo = load16(src), hi = load16(src + 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f[i] = as_f32(lo[i]);
          f[4 + i] = as_f32(hi[i]);
        }
      }
      dst += half * Sh::kHalf + s * 3 * kPsOperand;
    } else {                                 // V^T: channel 32b + c, keys 16j + (4g..4g+3, 8+4g..8+4g+3)
      const int o = op - 2 * Sh::kSteps;
      const int half = o / Sh::kSteps, j = o % Sh::kSteps / (kD / 32), b = o % (kD / 32);
      const int64_t key = key0 + half * 32 + j * 16 + 4 * g;
      const float *src = (const float *)a.v + h * a.v_head_stride + b * 32 + c;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int64_t tok = key + (i & 3) + (i >> 2) * 8;
        if (tok < S) f[i] = src[tok * a.v_tok_stride];
      }
      dst += Sh::kSide + half * Sh::kHalf + (j * (kD / 32) + b) * 3 * kPsOperand;
    }
    u32x4 part[3];
    split8(f, part);
#pragma unroll
    for (int i = 0; i < 8; ++i) bad |= !splits(f[i]);
#pragma unroll
    for (int i = 0; i < 3; ++i) store16(dst + i * kPsOperand, part[i]);
  }
  // the queries, which the attention kernel splits for itself
  const int64_t n_heads = (int64_t)a.rep * a.n_kv_heads;
  const int64_t n_vecs = S * n_heads * (kD / 4);
  for (int64_t i = (int64_t)blockIdx.x * kPsSplitThreads + threadIdx.x; i < n_vecs;
       i += (int64_t)gridDim.x * kPsSplitThreads) {
    const int64_t row = i / (kD / 4);
    const u32x4 v = load16(a.q + (row / n_heads * a.q_tok_stride + row % n_heads * a.q_head_stride) * 4 +
                           i % (kD / 4) * 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) bad |= !splits(as_f32(v[j]));
  }
  const int any = __syncthreads_or(bad);
  if (threadIdx.x == 0) flags[blockIdx.x] = any != 0;
}

template <int kD, int kHeads>
__global__ void __launch_bounds__(kPsThreads, 1)
prefill_attention_f32_split_kernel(const PrefillArgs a, const char *__restrict__ planes, const int64_t planes_rounds) {
  using Sh = SplitShape<kD>;
  constexpr int kBlockRows = 128 / kHeads;
  constexpr int kCBlocks = kD / 32;      // 32-channel blocks of O^T
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;
  const int c = lane & 31;
  __shared__ __align__(16) char smem[Sh::kBytes];

  if (prefill_gate(a)) return;           // (the splitting kernel met operands for the other kernel)

  // all heads' longest rows first, the kv heads in turn: see prefill_attention.hip
  const unsigned n_kv_heads = a.n_kv_heads;
  const unsigned piece = prefill_piece(a);
  const int hk = (int)(piece % n_kv_heads);
  const int64_t rem = piece / n_kv_heads;
  const int64_t rb = a.n_row_blocks - 1 - rem / a.n_groups;
  const int hq = hk * a.rep + (int)(rem % a.n_groups) * kHeads + (wave & 3) % kHeads;
  const int kgroup = wave >> 2;          // which 32 keys of a round
  const int64_t S = a.seq_len;
  const int64_t m0 = rb * kBlockRows;
  const int64_t row0 = m0 + (wave & 3) / kHeads * 32;
  const int64_t my_row = row0 + c;
  const int64_t last_key = (m0 + kBlockRows < S ? m0 + kBlockRows : S) - 1;
  const int n_rounds = (int)(last_key / kPsKeys) + 1;
  const int64_t wave_last_key = row0 + 31 < S ? row0 + 31 : S - 1;

  const char *src = planes + (int64_t)hk * planes_rounds * Sh::kRound + lane * 16;
  typedef __attribute__((address_space(1))) const void *GlobalPtr;
  typedef __attribute__((address_space(3))) void *LdsPtr;
  auto fetch_side = [&](int64_t from, int to) {
#pragma unroll
    for (int u = 0; u < Sh::kSide / kPsOperand / 8; ++u) {
      const int blk = wave + u * 8;
      __builtin_amdgcn_global_load_lds((GlobalPtr)(src + from + blk * kPsOperand),
                                       (LdsPtr)(smem + to + blk * kPsOperand), 16, 0, 0);
    }
  };
  auto fetch_k = [&](int round, int buf) { fetch_side((int64_t)round * Sh::kRound, buf * Sh::kSide); };
  auto fetch_v = [&](int round, int buf) {
    fetch_side((int64_t)round * Sh::kRound + Sh::kSide, (2 + (Sh::kVBufs == 2 ? buf : 0)) * Sh::kSide);
  };

  fetch_k(0, 0);
  if constexpr (Sh::kVBufs == 2) fetch_v(0, 0);

  // Q^T as the B operand: row c, channels 16s + 8g .. +7, in three parts
  u32x4 qf[Sh::kSteps][3];
  {
    const int64_t r = my_row < S ? my_row : S - 1;
    const char *qp = a.q + (r * a.q_tok_stride + (int64_t)hq * a.q_head_stride) * 4 + g * 32;
#pragma unroll
    for (int s = 0; s < Sh::kSteps; ++s) {
      const u32x4 lo = load16(qp + s * 64), hi = load16(qp + s * 64 + 16);
      float f[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f[i] = as_f32(lo[i]);
        f[4 + i] = as_f32(hi[i]);
      }
      split8(f, qf[s]);
    }
  }

  float m = kMinusHuge, l = 0.f;
  // [b]: channels 32b + 8j + 4g + i of row c in register 4j + i.  D 64 keeps the small products'
  // sums apart to the end; D 128 has no registers for that and adds a round's small
  // products and then its large ones up from zero before they join the output.
  constexpr bool kApart = kD == 64;
  ps_f32x16 acc[kCBlocks], small[kApart ? kCBlocks : 1];
#pragma unroll
  for (int b = 0; b < kCBlocks; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      acc[b][i] = 0.f;
      if (kApart) small[b][i] = 0.f;
    }

  u32x4 pt[2][3];   // P^T operands: [16 keys][part]
  auto scores = [&](int round, int buf, auto mask_tag) {
    constexpr bool kMask = decltype(mask_tag)::value;
    __builtin_amdgcn_iglp_opt(kD == 64);   // (measured: see the loop below)
    const char *kt = smem + buf * Sh::kSide + kgroup * Sh::kHalf + lane * 16;
    ps_f32x16 st, lo;
#pragma unroll
    for (int i = 0; i < 16; ++i) st[i] = lo[i] = 0.f;
#pragma unroll
    for (int s = 0; s < Sh::kSteps; ++s) {
      const u32x4 k1 = *(const u32x4 *)(kt + (3 * s) * kPsOperand);
      const u32x4 k2 = *(const u32x4 *)(kt + (3 * s + 1) * kPsOperand);
      const u32x4 k3 = *(const u32x4 *)(kt + (3 * s + 2) * kPsOperand);
      st = ps_mma(k1, qf[s][0], st);
      lo = ps_mma(k1, qf[s][2], lo);
      lo = ps_mma(k1, qf[s][1], lo);
      lo = ps_mma(k2, qf[s][1], lo);
      lo = ps_mma(k2, qf[s][0], lo);
      lo = ps_mma(k3, qf[s][0], lo);
    }
    st += lo;
    // register 4j + i: key 64 round + 32 kgroup + 8j + 4g + i
    if constexpr (kMask) {
      const int lim = (int)(my_row - ((int64_t)round * kPsKeys + kgroup * 32 + 4 * g));
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (8 * (i >> 2) + (i & 3) > lim) st[i] = -INFINITY;
    }
    float smax = st[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) smax = fmaxf(smax, st[i]);
    smax *= a.scale_log2;   // the scale is positive: max and scaling commute
    if (__any(smax > m + kRescaleSlack)) {  // rare after the first rounds
      float mx = fmaxf(m, smax);
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float alpha = fast_exp2(m - mx);
      m = mx;
      l *= alpha;
#pragma unroll
      for (int b = 0; b < kCBlocks; ++b) {
        acc[b] *= alpha;
        if (kApart) small[b] *= alpha;
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) st[i] = fast_exp2(fmaf(st[i], a.scale_log2, -m));
    l += (((st[0] + st[1]) + (st[2] + st[3])) + ((st[4] + st[5]) + (st[6] + st[7]))) +
         (((st[8] + st[9]) + (st[10] + st[11])) + ((st[12] + st[13]) + (st[14] + st[15])));
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float p[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] = st[8 * j + i] * kWeightScale;
      split8(p, pt[j]);
    }
  };
  auto values = [&](int buf) {
    __builtin_amdgcn_iglp_opt(kD == 64);
    const char *vt = smem + (2 + (Sh::kVBufs == 2 ? buf : 0)) * Sh::kSide + kgroup * Sh::kHalf + lane * 16;
    auto operand = [&](int j, int b, int part) {
      return *(const u32x4 *)(vt + ((j * kCBlocks + b) * 3 + part) * kPsOperand);
    };
    if constexpr (kApart) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int b = 0; b < kCBlocks; ++b) {
          const u32x4 v1 = operand(j, b, 0), v2 = operand(j, b, 1), v3 = operand(j, b, 2);
          acc[b] = ps_mma(v1, pt[j][0], acc[b]);
          small[b] = ps_mma(v1, pt[j][2], small[b]);
          small[b] = ps_mma(v1, pt[j][1], small[b]);
          small[b] = ps_mma(v2, pt[j][1], small[b]);
          small[b] = ps_mma(v2, pt[j][0], small[b]);
          small[b] = ps_mma(v3, pt[j][0], small[b]);
        }
    } else {
#pragma unroll
      for (int b = 0; b < kCBlocks; ++b) {
        ps_f32x16 sum;
#pragma unroll
        for (int i = 0; i < 16; ++i) sum[i] = 0.f;
        u32x4 v1[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          v1[j] = operand(j, b, 0);
          const u32x4 v2 = operand(j, b, 1), v3 = operand(j, b, 2);
          sum = ps_mma(v1[j], pt[j][2], sum);
          sum = ps_mma(v1[j], pt[j][1], sum);
          sum = ps_mma(v2, pt[j][1], sum);
          sum = ps_mma(v2, pt[j][0], sum);
          sum = ps_mma(v3, pt[j][0], sum);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) sum = ps_mma(v1[j], pt[j][0], sum);
        acc[b] += sum;
      }
    }
  };

  // A round out of buffers `buf`, the next one on its way into the others.
  auto whole_round = [&](int round, int buf, bool more, bool needed, auto mask_tag) {
    if constexpr (Sh::kVBufs == 2) {
      // the other buffers were last read before the barrier that ended the previous round
      if (more) {
        fetch_k(round + 1, buf ^ 1);
        fetch_v(round + 1, buf ^ 1);
      }
      if (needed) {
        scores(round, buf, mask_tag);
        values(buf);
      }
    } else {
      fetch_v(round, 0);                   // (V of the previous round was read before the last barrier)
      if (needed) scores(round, buf, mask_tag);
      __syncthreads();                     // V has landed
      if (more) fetch_k(round + 1, buf ^ 1);
      if (needed) values(0);
    }
    __syncthreads();                       // the next round has landed; everyone is done with this one
  };
  __syncthreads();
  // rounds that every wave needs whole, two at a time: constant LDS addresses.  iglp_opt(1) in both
  // halves of a round, which spreads the LDS reads between the MFMAs, gives D 64 1.5 % (9200 tokens, 8/2
  // heads: 472.7 -> 465.5 us) and takes 0.6 % at D 128, which has it off (iglp_opt(0)).
  const int n_whole = (int)(m0 / kPsKeys) & ~1;
  for (int round = 0; round < n_whole; round += 2) {
    whole_round(round, 0, true, true, std::false_type{});
    whole_round(round + 1, 1, true, true, std::false_type{});   // (there is a next one: the block's own rows)
  }
  for (int round = n_whole; round < n_rounds; ++round) {
    const int64_t t0 = (int64_t)round * kPsKeys + kgroup * 32;
    whole_round(round, round & 1, round + 1 < n_rounds, t0 <= wave_last_key, std::true_type{});
  }

  if constexpr (kApart) {
#pragma unroll
    for (int b = 0; b < kCBlocks; ++b) acc[b] += small[b];
  }
  // ---- the second group hands its state to the first, which merges and stores
  char *stash = smem + (wave & 3) * (kD / 8 + 1) * 1024 + lane * 16;
  if (kgroup == 1) {
#pragma unroll
    for (int b = 0; b < kCBlocks; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *(float4 *)(stash + (4 * b + j) * 1024) =
            make_float4(acc[b][4 * j], acc[b][4 * j + 1], acc[b][4 * j + 2], acc[b][4 * j + 3]);
    *(float2 *)(stash + 4 * kCBlocks * 1024) = make_float2(m, l);
  }
  __syncthreads();
  if (kgroup == 1) return;
  const float2 other = *(const float2 *)(stash + 4 * kCBlocks * 1024);
  const float mx = fmaxf(m, other.x);      // (finite: this group had key 0)
  const float mine = fast_exp2(m - mx), theirs = fast_exp2(other.x - mx);
  l = l * mine + other.y * theirs;
  l += __shfl_xor(l, 32, 64);
  const float inv = l > 0.f ? 1.f / l / kWeightScale : 0.f;
  if (my_row < S) {
    float *op = (float *)(a.out + (my_row * a.o_tok_stride + (int64_t)hq * a.o_head_stride) * 4) + 4 * g;
#pragma unroll
    for (int b = 0; b < kCBlocks; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4 o = *(const float4 *)(stash + (4 * b + j) * 1024);
        *(float4 *)(op + 32 * b + 8 * j) =
            make_float4((acc[b][4 * j] * mine + o.x * theirs) * inv, (acc[b][4 * j + 1] * mine + o.y * theirs) * inv,
                        (acc[b][4 * j + 2] * mine + o.z * theirs) * inv, (acc[b][4 * j + 3] * mine + o.w * theirs) * inv);
      }
    if (a.lse != nullptr && g == 0)
      a.lse[(int64_t)hq * S + my_row] = l > 0.f ? (mx + __builtin_amdgcn_logf(l)) * kLn2 : -INFINITY;
  }
}

template <int kD>
static int launch_prefill_f32_split(PrefillArgs a, char *workspace, hipStream_t s) {
  using Sh = SplitShape<kD>;
  const int heads = a.rep % 4 == 0 ? 4 : (a.rep % 2 == 0 ? 2 : 1);
  const int64_t rounds = ceil_div(a.seq_len, kPsKeys);
  const int64_t waves = rounds * 4 * Sh::kSteps * a.n_kv_heads;
  const int64_t want = ceil_div(waves, kPsSplitThreads / 64);
  const int split_blocks = (int)(want < kPsMaxSplitBlocks ? want : kPsMaxSplitBlocks);
  uint32_t *flags = (uint32_t *)workspace;
  char *planes = workspace + kPsMaxSplitBlocks * sizeof(uint32_t);
  hipLaunchKernelGGL(prefill_split_kernel<kD>, dim3(split_blocks), dim3(kPsSplitThreads), 0, s, a, planes, flags,
                     rounds);
  int rc = launch_status("da_prefill_attention_f32_split(split)");
  if (rc) return rc;
  a.gate = flags;
  a.n_gate = split_blocks;
  PrefillArgs b = a;
  b.n_groups = a.rep / heads;
  b.n_row_blocks = ceil_div(a.seq_len, 128 / heads);
  const int64_t blocks = b.n_row_blocks * b.n_groups * a.n_kv_heads;
  if (blocks > 0x7fffffff)
    return fail(DA_ENOTSUP, "da_prefill_attention_f32_split: %lld workgroups", (long long)blocks);
  prefill_order(b, blocks);
  const dim3 grid((unsigned)blocks);
  if (heads == 4)
    hipLaunchKernelGGL((prefill_attention_f32_split_kernel<kD, 4>), grid, dim3(kPsThreads), 0, s, b, planes, rounds);
  else if (heads == 2)
    hipLaunchKernelGGL((prefill_attention_f32_split_kernel<kD, 2>), grid, dim3(kPsThreads), 0, s, b, planes, rounds);
  else
    hipLaunchKernelGGL((prefill_attention_f32_split_kernel<kD, 1>), grid, dim3(kPsThreads), 0, s, b, planes, rounds);
  rc = launch_status("da_prefill_attention_f32_split");
  if (rc) return rc;
  a.gate_runs_if_set = 1;
  return launch_prefill_f32(a, kD, s);
}

static size_t split_workspace(int64_t seq_len, int n_kv_heads, int head_dim) {
  return kPsMaxSplitBlocks * sizeof(uint32_t) +
         (size_t)ceil_div(seq_len, kPsKeys) * n_kv_heads *
             (head_dim == 64 ? SplitShape<64>::kRound : SplitShape<128>::kRound);
}

// The plain kernel's one launch against the three here (10 us for splitting, 5 for the launch that
// returns at once, workgroups of twice the rows).  us, plain / split: D 64, any heads: 1000 tokens
// 46-48 / 47-52, 1200 55-61 / 53-59, 2000 88-112 / 81-90; D 128, by 2 S^2 Hq D: 8/2 heads 1400 tokens (4.0e9)
// 111 / 114, 1700 (5.9e9) 136 / 135; 24/8 800 (3.9e9) 76 / 73, 1000 (6.1e9) 101 / 90; 32/8 600 (2.9e9) 58 / 62,
// 1000 (8.2e9) 107 / 89; 64/8 600 (5.9e9) 66 / 65.
static bool split_pays(int64_t seq_len, int n_q_heads, int head_dim) {
  return head_dim == 64 ? seq_len >= 1200 : 2.0 * seq_len * seq_len * n_q_heads * head_dim >= 6e9;
}

}  // namespace da

extern "C" size_t da_prefill_attention_f32_workspace_bytes(int64_t seq_len, int n_q_heads, int n_kv_heads,
                                                           int head_dim) {
  using namespace da;
  if (seq_len <= 0 || n_kv_heads <= 0 || n_q_heads < n_kv_heads || n_q_heads % n_kv_heads ||
      (head_dim != 64 && head_dim != 128) || !split_pays(seq_len, n_q_heads, head_dim))
    return 0;
  return split_workspace(seq_len, n_kv_heads, head_dim);
}

extern "C" int da_prefill_attention_f32_split(const float *q, int64_t q_tok_stride, int64_t q_head_stride,
                                              const float *k, int64_t k_tok_stride, int64_t k_head_stride,
                                              const float *v, int64_t v_tok_stride, int64_t v_head_stride,
                                              int64_t seq_len, int n_q_heads, int n_kv_heads, int head_dim,
                                              float scale, float *out, int64_t o_tok_stride,
                                              int64_t o_head_stride, float *lse_out, void *workspace,
                                              size_t workspace_bytes, void *stream) {
  using namespace da;
  PrefillArgs a = {};
  const int rc = prefill_args(a, "da_prefill_attention_f32_split", q, q_tok_stride, q_head_stride, k, k_tok_stride,
                              k_head_stride, v, v_tok_stride, v_head_stride, seq_len, n_q_heads, n_kv_heads,
                              DA_F32, scale, out, o_tok_stride, o_head_stride, lse_out);
  if (rc != DA_OK || seq_len == 0) return rc;
  if (head_dim != 64 && head_dim != 128)
    return fail(DA_ENOTSUP, "da_prefill_attention_f32_split: head_dim 64 or 128 (got %d)", head_dim);
  const size_t need = split_workspace(seq_len, n_kv_heads, head_dim);
  DA_REQUIRE(workspace && (uintptr_t)workspace % 16 == 0 && workspace_bytes >= need,
             "da_prefill_attention_f32_split: %zu bytes of 16-byte aligned workspace needed", need);
  return head_dim == 128 ? launch_prefill_f32_split<128>(a, (char *)workspace, (hipStream_t)stream)
                         : launch_prefill_f32_split<64>(a, (char *)workspace, (hipStream_t)stream);
}
