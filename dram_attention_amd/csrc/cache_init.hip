// Initial metadata of a page cache: step 0, no access yet, slot s holding page first + s.
// Counterpart of the buffers LRUCache.__init__ of the reference fills with torch
// operators, dram_attention/lru_cache.py:143-189.
//
// One launch instead of eight fills and copies of 5 us each ahead of every prompt's
// attention (and the host work that issues them): the fp32 layer's 9200 tokens 948 -> 911 us,
// two model layers' 8192 tokens 6.55 -> 6.47 ms.
#include "page_minmax.hpp"

namespace da {

__device__ __forceinline__ void page_cache_item(int32_t *__restrict__ step, float *__restrict__ access_time,
                                                int64_t *__restrict__ d2h, int64_t *__restrict__ h2d, int n_heads,
                                                int64_t n_pages, int64_t n_slots, int64_t first, int64_t i) {
  if (i == 0) *step = 0;
  if (i < n_pages * n_heads) {
    const int64_t slot = i % n_pages - first;
    d2h[i] = slot >= 0 ? slot : -1;
  }
  if (i < n_slots * n_heads) {
    access_time[i] = 0.f;
    h2d[i] = i % n_slots + first;
  }
}

__global__ void __launch_bounds__(256)
page_cache_init_kernel(int32_t *__restrict__ step, float *__restrict__ access_time, int64_t *__restrict__ d2h,
                       int64_t *__restrict__ h2d, int n_heads, int64_t n_pages, int64_t n_slots, int64_t first) {
  page_cache_item(step, access_time, d2h, h2d, n_heads, n_pages, n_slots, first, (int64_t)blockIdx.x * 256 + threadIdx.x);
}

// What a prompt leaves behind besides its page store, as one launch: the page summaries (workgroups
// [0, minmax_blocks)), the metadata of the page cache and the local window's copy of the last tokens.  Bound:
// HBM for the summaries, launches for the rest: four of them in a row, 12 + 5 + 5.5 + 5.5 us behind the
// attention of 9200 tokens in fp32, whatever their size; a static prefix has the two copies only.
// us a prompt, the separate launches / this one (two runs of one side differ by up to 0.4 %): 9200 tokens of 8/2 heads in
// fp32 473.3 / 465.2; no difference shown for 8192 through two layers of a model (6366 / 6357) and 4613 of
// 32/8, a static prefix (173.7 / 173.0).
struct PromptCacheArgs {
  const char *k, *v;                  // (tokens, heads, head_dim)
  int64_t tok_stride, head_stride;    // elements
  int n_heads, vecs_per_row, page;
  int64_t n_pages, n_slots;
  char *summaries;
  int minmax_blocks;
  int32_t *step;                      // null: no page cache
  float *access_time;
  int64_t *d2h, *h2d;
  char *window_k, *window_v;          // the tokens behind the pages
  int64_t window_vecs;                // 16-byte lanes of each
};
template <typename T>
__global__ void __launch_bounds__(256)
prompt_cache_kernel(const PromptCacheArgs a) {
  const int b = blockIdx.x;
  if (b < a.minmax_blocks) {
    page_minmax_vec<T>(a.k, a.head_stride, a.tok_stride, a.n_heads, a.n_pages, a.page, a.vecs_per_row, a.summaries,
                       (int64_t)b * 256 + threadIdx.x, (int64_t)a.minmax_blocks * 256);
    return;
  }
  const int64_t i = (int64_t)(b - a.minmax_blocks) * 256 + threadIdx.x;
  if (a.step != nullptr)
    page_cache_item(a.step, a.access_time, a.d2h, a.h2d, a.n_heads, a.n_pages, a.n_slots, a.n_pages - a.n_slots, i);
  if (i < a.window_vecs) {
    const int64_t row = i / a.vecs_per_row, c = i % a.vecs_per_row;
    const int64_t tok = a.n_pages * a.page + row / a.n_heads;
    const int64_t at = (tok * a.tok_stride + row % a.n_heads * a.head_stride) * T::kBytes + c * 16;
    const u32x4 k = load16(a.k + at), v = load16(a.v + at);
    store16(a.window_k + i * 16, k);
    store16(a.window_v + i * 16, v);
  }
}

}  // namespace da

extern "C" int da_page_cache_init(int32_t *current_step, float *access_time, int64_t *dram_to_hbm,
                                  int64_t *hbm_to_dram, int n_kv_heads, int64_t n_pages, int64_t n_slots,
                                  void *stream) {
  using namespace da;
  DA_REQUIRE(n_kv_heads >= 0 && n_slots >= 0 && n_pages >= n_slots, "da_page_cache_init: bad geometry");
  DA_REQUIRE(current_step && (access_time && hbm_to_dram || n_slots * n_kv_heads == 0) &&
                 (dram_to_hbm || n_pages * n_kv_heads == 0),
             "da_page_cache_init: null pointer");
  const int64_t items = n_pages * n_kv_heads > 0 ? n_pages * n_kv_heads : 1;
  if (ceil_div(items, 256) > 0x7fffffff) return fail(DA_ENOTSUP, "da_page_cache_init: too many pages");
  hipLaunchKernelGGL(page_cache_init_kernel, dim3((unsigned)ceil_div(items, 256)), dim3(256), 0,
                     (hipStream_t)stream, current_step, access_time, dram_to_hbm, hbm_to_dram, n_kv_heads, n_pages,
                     n_slots, n_pages - n_slots);
  return launch_status("da_page_cache_init");
}

extern "C" int da_prompt_cache(const void *k, const void *v, int64_t tok_stride, int64_t head_stride, int64_t n_tokens,
                               int n_kv_heads, int head_dim, int dtype, int64_t n_pages, int page_size,
                               int64_t n_slots, void *summaries, int32_t *current_step, float *access_time,
                               int64_t *dram_to_hbm, int64_t *hbm_to_dram, void *window_k, void *window_v,
                               void *stream) {
  using namespace da;
  DA_REQUIRE(dtype == DA_F32 || dtype == DA_F16 || dtype == DA_BF16, "da_prompt_cache: unknown dtype %d", dtype);
  DA_REQUIRE(n_kv_heads > 0 && head_dim > 0 && page_size > 0 && n_pages >= 0 && n_pages <= n_tokens / page_size &&
                 n_slots >= 0 && n_slots <= n_pages,
             "da_prompt_cache: bad geometry");
  const bool paged = current_step != nullptr;
  const int64_t window = n_tokens - n_pages * page_size;
  DA_REQUIRE(k && v && (window == 0 || (window_k && window_v)), "da_prompt_cache: null pointer");
  DA_REQUIRE(!paged || (summaries && dram_to_hbm && n_pages > 0 && (n_slots == 0 || (access_time && hbm_to_dram))),
             "da_prompt_cache: null pointer of a page cache, or none of its pages");
  const int vec = 16 / elem_size(dtype);
  DA_REQUIRE(minmax_vec_fits(k, head_stride, tok_stride, head_dim, dtype, summaries) && (uintptr_t)v % 16 == 0 &&
                 (uintptr_t)window_k % 16 == 0 && (uintptr_t)window_v % 16 == 0,
             "da_prompt_cache: rows must be 16-byte aligned");
  PromptCacheArgs a = {};
  a.k = (const char *)k;
  a.v = (const char *)v;
  a.tok_stride = tok_stride;
  a.head_stride = head_stride;
  a.n_heads = n_kv_heads;
  a.vecs_per_row = head_dim / vec;
  a.page = page_size;
  a.n_pages = n_pages;
  a.n_slots = n_slots;
  a.window_k = (char *)window_k;
  a.window_v = (char *)window_v;
  a.window_vecs = window * n_kv_heads * a.vecs_per_row;
  int64_t items = a.window_vecs;
  if (paged) {
    a.summaries = (char *)summaries;
    a.step = current_step;
    a.access_time = access_time;
    a.d2h = dram_to_hbm;
    a.h2d = hbm_to_dram;
    const int64_t blocks = ceil_div(n_pages * n_kv_heads * a.vecs_per_row, 256);
    a.minmax_blocks = (int)(blocks < 65536 ? blocks : 65536);
    if (n_pages * n_kv_heads > items) items = n_pages * n_kv_heads;
  }
  if (items == 0) return DA_OK;
  if (ceil_div(items, 256) > 0x3fffffff) return fail(DA_ENOTSUP, "da_prompt_cache: too many tokens");
  const dim3 grid((unsigned)(a.minmax_blocks + ceil_div(items, 256)));
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case DA_F32: hipLaunchKernelGGL(prompt_cache_kernel<F32>, grid, dim3(256), 0, s, a); break;
    case DA_F16: hipLaunchKernelGGL(prompt_cache_kernel<F16>, grid, dim3(256), 0, s, a); break;
    default: hipLaunchKernelGGL(prompt_cache_kernel<BF16>, grid, dim3(256), 0, s, a);
  }
  return launch_status("da_prompt_cache");
}
