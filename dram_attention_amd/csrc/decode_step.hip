// One decode step of one layer as one call: page scores, ordered top-k with the list of
// least recent slots, LRU update, then page stream, attention and merge (the sequence of
// DRAMAttention.forward's generate stage, dram_attention/dram_attention.py:144-238 of the
// reference).  Host code only: it issues the launches of the entry points it stands for, on the
// operands of one argument block, selection and LRU update as one where their sizes allow.
//
// What it saves is the caller's time: five calls of 18 to 33 arguments take 86 us to marshal from
// Python, where a step of the small layers takes 25 us of the GPU.  Five calls / this one: the fp32
// layer over 8K tokens 85 / 34 us a step, four 2048-wide model layers launched from Python
// 674 / 435 us a token (25 and 277 since, by what the one call is made of).
//
// Several layers whose queries do not depend on each other (da_decode_steps): all scores in a
// launch, all selections and updates in a launch, all page streams in a launch
// (stream_attention.hip), all merges in a launch, eight layers at a time.  The stream of a layer waits for the host link and everything else is a chain of short
// launches; a second queue that takes the chains of the other layers beside the stream hides them,
// but each hand-over between queues of a graph idles 9 us and a selection beside a stream takes
// three times as long and slows it.  us a model step in one graph, two queues / this: 4 layers of
// 64K tokens, 32/8 heads 363 / 302 (309 with a launch of scores per layer); 4 of 128K 612 / 561; 3 of 250K
// 391 / 356; 5 of 12K, 28/4 217 / 115 (130); 4 of 20K, 16/16, D 64 153 / 89 (96); 2 of 8K, 16/4, D 64 87 / 45 (48).
#include "page_stream.hpp"
#include "topk_rows.hpp"

namespace da {

static int check_step(const da_decode_step_args &a) {
  DA_REQUIRE(a.n_q_heads > 0 && a.n_kv_heads > 0 && a.n_q_heads % a.n_kv_heads == 0 && a.kp > 0 &&
                 a.page_size > 0 && a.n_slots >= 0,
             "da_decode_step: bad geometry");
  return DA_OK;
}

// What da_page_score refuses of a step that check_step and prepare_step let pass.
static int check_scores(const da_decode_step_args &a) {
  DA_REQUIRE(a.minmax && a.scores, "da_decode_step: null pointer");
  DA_REQUIRE((a.score_flags & ~(DA_SCORE_ROUND | DA_SCORE_ORDERED_BOUNDS)) == 0,
             "da_decode_step: unknown score flag bits %d", a.score_flags);
  return DA_OK;
}

static int scores_of(const da_decode_step_args &a, void *stream) {
  const int H = a.n_kv_heads, D = a.head_dim, rep = a.n_q_heads / H;
  return da_page_score(a.q, a.q_head_stride, a.q_head_stride * rep, a.minmax, a.n_pages * 2 * D, 2 * D, D, rep, H,
                       a.n_pages, D, a.dtype, a.scores, (int64_t)H * a.n_pages, a.n_pages, DA_F32, a.score_flags,
                       stream);
}

// (Rows of more than 4096 pages keep the two launches: their steps stream for so long that the caller's
// time is hidden, and on the GPU the hand-over is 0.4 us slower there than a launch: 128K tokens 160.8 /
// 161.5 us; 3064 pages 81.2 / 81.0.  Rows of up to 2048 pages are select_short.hip's in most cases.)
static int select_and_update(const da_decode_step_args &a, void *stream) {
  if (a.n_pages <= 4096 && topk_lru_in_one_launch(a)) return launch_topk_lru(&a, 1, (hipStream_t)stream);
  const int H = a.n_kv_heads, rep = a.n_q_heads / H, K = rep * a.kp;
  const int rc = da_topk_pages_lru(a.scores, (int64_t)H * a.n_pages, a.n_pages, rep, rep, H, a.n_pages, a.kp, a.idx, K,
                                   K, a.kp, DA_I64, a.access_time, a.n_slots, DA_TIME_F32, a.n_slots, a.k_cand,
                                   a.candidates, a.step, a.topk_workspace, a.topk_workspace_bytes, stream);
  if (rc) return rc;
  return da_lru_update(a.idx, K, DA_I64, H, K, a.n_pages, a.n_slots, a.step, DA_LRU_BUMP_STEP, a.access_time,
                       a.n_slots, DA_TIME_F32, a.d2h, a.n_pages, a.h2d, a.n_slots, DA_I64, a.hit_mask, a.miss_page,
                       a.miss_slot, a.miss_count, a.slot_epoch, a.candidates, a.k_cand, a.lru_workspace,
                       a.lru_workspace_bytes, stream);
}

static da_paged_overlap overlap_of(const da_decode_step_args &a, int phase) {
  const int64_t e = elem_size(a.dtype), page = (int64_t)a.page_size * 2 * a.head_dim;
  da_paged_overlap o = {};
  o.page_size = a.page_size;
  o.phase = phase;
  o.slot_epoch = a.slot_epoch;
  o.slot_epoch_head_stride = a.n_slots;
  o.epoch = a.step;
  o.miss_slot = a.miss_slot;
  o.miss_count = a.miss_count;
  o.miss_capacity = a.n_q_heads / a.n_kv_heads * a.kp;
  o.gather_blocks = a.gather_blocks;
  o.dram = a.dram;
  o.dram_head_stride_bytes = a.n_pages * page * e;
  o.dram_page_stride_bytes = page * e;
  o.hbm = a.hbm;
  o.hbm_head_stride_bytes = a.n_slots * page * e;
  o.hbm_slot_stride_bytes = page * e;
  o.miss_page = a.miss_page;
  o.link_gbps = a.link_gbps;
  o.block_gbps = a.block_gbps;
  return o;
}

static int stream_and_attend(const da_decode_step_args &a, int phase, void *stream) {
  const int H = a.n_kv_heads, D = a.head_dim;
  const da_paged_overlap o = overlap_of(a, phase);
  const char *hbm = (const char *)a.hbm;
  return da_decode_attention_paged(
      a.q, a.q_head_stride, a.n_q_heads, H, D, a.dtype, hbm, hbm + D * elem_size(a.dtype), 2 * D,
      (int64_t)a.n_slots * a.page_size * 2 * D, (int64_t)a.n_slots * a.page_size, a.cache_k, a.cache_v, (int64_t)H * D,
      D, a.cache_rows, a.cache_len, a.cache_len_dev, a.new_k, a.new_v, D, a.scale, a.out, D, nullptr, a.workspace,
      a.workspace_bytes, &o, stream);
}

static int prepare_step(const da_decode_step_args &a, PreparedAttention &p) {
  const int H = a.n_kv_heads, D = a.head_dim;
  const da_paged_overlap o = overlap_of(a, DA_PHASE_STREAM | DA_PHASE_FIRST);
  const char *hbm = (const char *)a.hbm;
  return prepare_attention(
      a.q, a.q_head_stride, a.n_q_heads, H, D, a.dtype, hbm, hbm + D * elem_size(a.dtype), 2 * D,
      (int64_t)a.n_slots * a.page_size * 2 * D, (int64_t)a.n_slots * a.page_size, a.cache_k, a.cache_v, (int64_t)H * D,
      D, a.cache_rows, a.cache_len, a.cache_len_dev, a.new_k, a.new_v, D, a.scale, a.out, a.workspace,
      a.workspace_bytes, &o, p);
}

// Whether two steps differ in nothing but their operands' places.
static bool same_sizes(const da_decode_step_args &a, const da_decode_step_args &b) {
  return a.n_q_heads == b.n_q_heads && a.n_kv_heads == b.n_kv_heads && a.head_dim == b.head_dim &&
         a.dtype == b.dtype && a.page_size == b.page_size && a.kp == b.kp && a.n_slots == b.n_slots &&
         a.k_cand == b.k_cand && a.gather_blocks == b.gather_blocks && a.n_pages == b.n_pages &&
         a.cache_rows == b.cache_rows;
}

}  // namespace da

extern "C" int da_decode_step(const da_decode_step_args *a, size_t args_bytes, void *stream) {
  using namespace da;
  DA_REQUIRE(a && args_bytes == sizeof(*a), "da_decode_step: argument block of %zu bytes, expected %zu",
             args_bytes, sizeof(*a));
  int rc = check_step(*a);
  if (rc) return rc;
  rc = scores_of(*a, stream);
  if (rc) return rc;
  rc = select_and_update(*a, stream);
  if (rc) return rc;
  return stream_and_attend(*a, DA_PHASE_STREAM | DA_PHASE_FIRST | DA_PHASE_SECOND, stream);
}

extern "C" int da_decode_steps_supported(const da_decode_step_args *a, int n_steps, size_t args_bytes) {
  using namespace da;
  if (!a || n_steps < 1 || args_bytes != n_steps * sizeof(*a)) return 0;
  for (int i = 0; i < n_steps; ++i)
    if (check_step(a[i]) != DA_OK || !same_sizes(a[i], a[0]) || !topk_lru_in_one_launch(a[i])) return 0;
  return 1;
}

extern "C" int da_decode_steps(const da_decode_step_args *a, int n_steps, size_t args_bytes, void *stream) {
  using namespace da;
  DA_REQUIRE(a && n_steps >= 1 && args_bytes == n_steps * sizeof(*a),
             "da_decode_steps: argument blocks of %zu bytes, expected %d of %zu", args_bytes, n_steps, sizeof(*a));
  if (!da_decode_steps_supported(a, n_steps, args_bytes))
    return fail(DA_ENOTSUP, "da_decode_steps: layers of the same sizes, whose selection and update are one launch");
  PreparedAttention p[kStepBatch];
  for (int i = 0; i < n_steps; ++i) {     // (every operand of every block is looked at before the first launch)
    int rc = prepare_step(a[i], p[0]);
    if (rc == DA_OK) rc = check_scores(a[i]);
    if (rc == DA_OK) rc = check_topk_lru(a[i]);
    if (rc) return rc;
  }
  hipStream_t s = (hipStream_t)stream;
  for (; n_steps > 0; a += kStepBatch, n_steps -= kStepBatch) {
    const int n = n_steps < kStepBatch ? n_steps : kStepBatch;
    int rc = DA_OK;
    for (int i = 0; i < n && rc == DA_OK; ++i) rc = prepare_step(a[i], p[i]);
    if (rc) return rc;
    bool scored = false;
    rc = launch_score_layers(a, n, &scored, s);
    for (int i = 0; i < n && rc == DA_OK && !scored; ++i) rc = scores_of(a[i], stream);
    if (rc) return rc;
    rc = launch_topk_lru(a, n, s);
    if (rc) return rc;
    if (stream_layers_supported(p[0])) {
      rc = launch_stream_layers(p, n, s);
    } else {
      for (int i = 0; i < n && rc == DA_OK; ++i) rc = stream_and_attend(a[i], DA_PHASE_STREAM | DA_PHASE_FIRST, stream);
    }
    if (rc) return rc;
    rc = launch_merge_layers(p, a, n, s);
    if (rc) return rc;
  }
  return DA_OK;
}
