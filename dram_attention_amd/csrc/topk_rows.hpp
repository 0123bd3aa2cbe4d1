// Rows of the page selection and the list of least recent slots that rides with them, as blocks
// of a launch: shared by the selection alone (topk_pages.hip) and the one that the LRU update
// follows in the same launch (lru_update.hip).
#pragma once

#include "lru_keys.hpp"

namespace da {

// Accesses to what other workgroups of the same launch wrote or will read (kShared): each die
// has an L2 of its own, so these go through to the memory behind them.
template <bool kShared, typename T>
__device__ __forceinline__ T load_between(const T *p) {
  if constexpr (kShared) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else return *p;
}
template <bool kShared, typename T>
__device__ __forceinline__ void store_between(T *p, T v) {
  if constexpr (kShared) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}

struct ScoreKey {
  const float *row;
  bool aligned;  // row starts on a 16-byte boundary
  __device__ __forceinline__ uint32_t operator()(int i) const { return float_order_key(row[i]); }
  __device__ __forceinline__ void load4(int i, uint32_t *k) const {
    float4 v;
    if (aligned) {
      v = *(const float4 *)(row + i);
    } else {
      v = make_float4(row[i], row[i + 1], row[i + 2], row[i + 3]);
    }
    k[0] = float_order_key(v.x);
    k[1] = float_order_key(v.y);
    k[2] = float_order_key(v.z);
    k[3] = float_order_key(v.w);
  }
};

// The k_cand least recently used slots of kv head h, in eviction order, into
// out[h, 0..k_cand).  Independent of this step's scores, so it rides along with
// the top-k launch (one more workgroup per head) and the LRU update that follows
// only has to drop the slots it touched from this list.
struct LruCandidateArgs {
  const void *access_time;  // (Hkv, n_slots), fp32 or int32; null: no candidates
  int64_t time_head_stride;
  int time_is_i32;
  int n_slots, k_cand;
  int32_t *out;  // (Hkv, k_cand) lists, then Hkv stamp words
  const int32_t *step;  // the LRU step counter: its value now is the list's stamp
  int n_heads;
};

template <bool kShared, typename TimeT>
__device__ __forceinline__ void lru_candidates_block(const LruCandidateArgs &c, int h,
                                                     SelectShared &sm) {
  LeastRecentKey<TimeT> key{(const TimeT *)c.access_time + h * c.time_head_stride};
  int32_t *dst = c.out + (int64_t)h * c.k_cand;
  // The stamp says which state of the access times the list describes: the update
  // that consumes the list compares it with the step it reads.
  if (threadIdx.x == 0) store_between<kShared>(c.out + (int64_t)c.n_heads * c.k_cand + h, *c.step);
  select_sorted(key, c.n_slots, c.k_cand, sm,
                direct([=](uint32_t rank, uint32_t slot) { store_between<kShared>(dst + rank, (int32_t)slot); }));
}

// Ordered top-k of every row, the list of least recent slots and the LRU update of a decode step
// as one launch (lru_update.hip).  Whether a step's sizes allow it, whether its operands are there, and
// the launch itself, which checks them too, of n <= kStepBatch layers of the same sizes.
constexpr int kStepBatch = 8;
bool topk_lru_in_one_launch(const da_decode_step_args &a);
int check_topk_lru(const da_decode_step_args &a);
int launch_topk_lru(const da_decode_step_args *a, int n, hipStream_t s);
// The same for short rows, a workgroup per kv head (select_short.hip); the operands are checked.
bool topk_lru_short(const da_decode_step_args &a);
int launch_topk_lru_short(const da_decode_step_args *a, int n, hipStream_t s);

// The page scores of those layers (page_score.hip).
int launch_score_layers(const da_decode_step_args *a, int n, bool *done, hipStream_t s);

}  // namespace da
