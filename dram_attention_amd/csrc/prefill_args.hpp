// Arguments of the causal prefill kernels (prefill_attention.hip for the 16-bit types,
// prefill_attention_f32.hip) and the checks their entry points share.
#pragma once
#include "attention_core.hpp"

namespace da {

struct PrefillArgs {
  const char *q, *k, *v;
  char *out;
  float *lse;  // (Hq, S) natural log, or null
  int64_t q_tok_stride, q_head_stride;  // elements
  int64_t k_tok_stride, k_head_stride;
  int64_t v_tok_stride, v_head_stride;
  int64_t o_tok_stride, o_head_stride;
  int64_t seq_len;
  int rep;          // query heads per kv head
  int n_groups;     // workgroups that share a kv head's rows: rep / kHeads
  int64_t n_row_blocks;
  int n_kv_heads;
  int late_at, n_late;  // the last n_late pieces of work take the places from late_at on (0: in order)
  float scale_log2;
  // fp32 only: words of which one is not zero where the prompt's operands do not split into three
  // bf16 parts (null: nobody looked); the plain kernel then runs if gate_runs_if_set, the split one if not
  const uint32_t *gate;
  int n_gate;
  int gate_runs_if_set;
};

// Whether this launch is not the one that does the prompt (the whole workgroup calls it).
__device__ __forceinline__ bool prefill_gate(const PrefillArgs &a) {
  if (a.gate == nullptr) return false;
  uint32_t any = 0;
  for (int i = threadIdx.x; i < a.n_gate; i += blockDim.x) any |= a.gate[i];
  return (__syncthreads_or((int)any) != 0) != (a.gate_runs_if_set != 0);
}

// Which piece of work, numbered longest first, a workgroup takes.  With one workgroup per compute
// unit, pieces go in grid order to the first unit that is free; workgroups are dealt in turn to the
// part's 32 shader engines before that, so an engine's eight units share every 32nd.  Longest first,
// the second 256 pieces pair up with the first, longest with shortest, to sums that are all alike, and
// if there are two rounds and a part of one, the short pieces of the third prolong as many units.  So those
// go ahead of the second round and in place of the shortest pieces of the first: the units that take
// them have time for three.  By 32s, which keeps every engine's share and which head a die works on.
// us in order / like this, D 128: 4613 tokens of 32/8 heads (584 pieces) 176 / 170, 5200 (656) 222 / 210, 6000
// (752) 284 / 272; 3600, 40/10 (570) 137 / 131; 2300, 64/8 (576) 94.4 / 87.2; D 64: 10000, 16/4 (628) 246 / 230.  Four
// rounds and a part gain 1 to 3 % (8700 tokens, 1088 pieces 561 / 552; 9200, 1152 628 / 611); three lose as
// much as they gain, and a part of less than 32 is not worth it (4613 of 28/4, 532: 159 / 161).
__device__ __forceinline__ unsigned prefill_piece(const PrefillArgs &a) {
  const unsigned b = blockIdx.x, at = a.late_at, n = a.n_late;
  return b < at || n == 0 ? b : b < at + n ? gridDim.x - n + (b - at) : b - n;
}
inline void prefill_order(PrefillArgs &a, int64_t pieces) {
  constexpr int kUnits = 256, kEngines = 32;
  const int rounds = (int)(pieces / kUnits < 8 ? pieces / kUnits : 8), part = (int)(pieces % kUnits);
  a.n_late = 0;
  if ((rounds != 2 && rounds != 4) || part <= kEngines) return;
  const int n = (int)ceil_div(part, kEngines), ahead = ((rounds == 2 ? 6 : 5) * n + 5) / 10;
  a.n_late = n * kEngines;
  a.late_at = kUnits - ahead * kEngines;
}

// The kernel on fp32 instructions (prefill_attention_f32.hip), head_dim 64 or 128.
int launch_prefill_f32(const PrefillArgs &a, int head_dim, hipStream_t s);

// Checks the operands of a prefill call and fills `a` (all but the grid's geometry).
inline int prefill_args(PrefillArgs &a, const char *what, const void *q, int64_t q_tok_stride,
                        int64_t q_head_stride, const void *k, int64_t k_tok_stride, int64_t k_head_stride,
                        const void *v, int64_t v_tok_stride, int64_t v_head_stride, int64_t seq_len,
                        int n_q_heads, int n_kv_heads, int dtype, float scale, void *out,
                        int64_t o_tok_stride, int64_t o_head_stride, float *lse_out) {
  DA_REQUIRE(n_q_heads > 0 && n_kv_heads > 0 && n_q_heads % n_kv_heads == 0,
             "%s: %d query heads do not split over %d kv heads", what, n_q_heads, n_kv_heads);
  DA_REQUIRE(seq_len >= 0, "%s: negative length", what);
  DA_REQUIRE(dtype == DA_F32 || dtype == DA_F16 || dtype == DA_BF16, "%s: unknown dtype %d", what, dtype);
  DA_REQUIRE(scale > 0.f, "%s: the softmax scale must be positive", what);
  if (seq_len == 0) return DA_OK;
  DA_REQUIRE(q && k && v && out, "%s: null pointer", what);
  const int64_t e = elem_size(dtype);
  for (int64_t stride : {q_tok_stride, q_head_stride, k_tok_stride, k_head_stride, v_tok_stride, v_head_stride,
                         o_tok_stride, o_head_stride})
    DA_REQUIRE(stride * e % 16 == 0, "%s: rows must be 16-byte aligned", what);
  DA_REQUIRE((uintptr_t)q % 16 == 0 && (uintptr_t)k % 16 == 0 && (uintptr_t)v % 16 == 0 && (uintptr_t)out % 16 == 0,
             "%s: rows must be 16-byte aligned", what);
  // (a tile's byte offsets from its first row are formed in 32 bits)
  const int64_t most = ((int64_t)1 << 24) / e;
  if (k_tok_stride < 0 || v_tok_stride < 0 || k_tok_stride > most || v_tok_stride > most)
    return fail(DA_ENOTSUP, "%s: key/value token strides of 0..2^24 bytes", what);
  a.q = (const char *)q;
  a.k = (const char *)k;
  a.v = (const char *)v;
  a.out = (char *)out;
  a.lse = lse_out;
  a.q_tok_stride = q_tok_stride;
  a.q_head_stride = q_head_stride;
  a.k_tok_stride = k_tok_stride;
  a.k_head_stride = k_head_stride;
  a.v_tok_stride = v_tok_stride;
  a.v_head_stride = v_head_stride;
  a.o_tok_stride = o_tok_stride;
  a.o_head_stride = o_head_stride;
  a.seq_len = seq_len;
  a.rep = n_q_heads / n_kv_heads;
  a.n_kv_heads = n_kv_heads;
  a.scale_log2 = scale * kLog2e;
  return DA_OK;
}

}  // namespace da
