// Initial metadata of a page cache: step 0, no access yet, slot s holding page first + s.
// Counterpart of the buffers LRUCache.__init__ of the reference fills with torch
// operators, dram_attention/lru_cache.py:143-189.
//
// One launch instead of eight fills and copies of 5 us each ahead of every prompt's
// attention (and the host work that issues them): the fp32 layer's 9200 tokens 948 -> 911 us,
// two model layers' 8192 tokens 6.55 -> 6.47 ms.
#include "common.hpp"

namespace da {

__global__ void __launch_bounds__(256)
page_cache_init_kernel(int32_t *__restrict__ step, float *__restrict__ access_time, int64_t *__restrict__ d2h,
                       int64_t *__restrict__ h2d, int n_heads, int64_t n_pages, int64_t n_slots, int64_t first) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
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
