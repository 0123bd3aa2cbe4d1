// Ordered top-k of a kv head's score rows and the LRU update it feeds, for short rows: one
// workgroup does a whole head.  The same results as topk_lru_update_kernel (lru_update.hip), which
// puts every row on a workgroup of its own and hands the lists over through memory.
//
// Bound: latency, a chain of dependent steps over a few KB.  What counts is how few of them
// there are and that they stay inside a wave or, at worst, inside the workgroup:
//   - a wave selects a row, its keys in registers (key j*64 + lane in register j): the k-th largest by
//     histograms of eight bits from the highest in which two keys differ (bf16 scores: two at
//     most; it ends as soon as a whole bin is wanted), the survivors compacted by every lane for
//     itself and ordered by counting, without one barrier;
//   - another wave meanwhile puts all slots in order of their access times by a stable radix
//     sort that only it takes part in, so the list of least recent slots is complete;
//   - both page maps are in LDS by then (a short row has few pages): the update reads nothing
//     from memory but the ticket of the step counter, with one thread per request and one per slot.
// us a launch (under the profiler; in brackets a workgroup a row): 512 pages of 2 heads in fp32, 4 rows of
// 32 pages, 128 slots 5.9 (12.9); 445 of 4 heads in bf16, the same lists 6.2 (12.0); 1000 of 8 heads, 4 rows of 64,
// 256 slots 7.3 (12.1), of 128, 512 slots 9.4 (13.3); 8 rows of 60 10.8 (13.6); 2047 of 8 heads, 4 rows of 128, 512
// slots 10.5 (13.1); fp32, 100 of 1000 pages 8.7 (13.5), 120 of 1800, 900 slots 12.3 (14.0).  Bisection bit by bit
// in place of the histograms: 6.4 for the first, 13.0 for 2047 pages.
//
// The rule (topk_lru_short): rows of at most 2048 pages (32 registers of keys), 8 rows a head, lists of
// 128 pages (ordering by counting grows with the square), 1024 requests and 1024 slots (a thread each);
// of the slots no more than 896 where the row is longer than 1024 pages: the one wave that sorts them
// is the last to be done there (1800 pages, 7 rows of 100, 1000 slots 13.5 (13.3)).
#include <type_traits>

#include "topk_rows.hpp"

namespace da {

constexpr int kShortPages = 2048, kShortRows = 8, kShortList = 128;
constexpr int kShortSlots = kSelThreads;
constexpr int kShortSlotRegs = kShortSlots / 64;
constexpr int kSlotWave = kSelWaves - 1;   // the wave that orders the slots
static_assert(kShortRows <= kSlotWave, "rows and slots on different waves");

typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));

struct ShortLayer {
  const float *scores;  // (rows, heads, pages)
  int n_rows, n_pages, kp, n_slots, k_cand;
  int64_t *idx;         // (heads, rows * kp)
  float *time;
  int64_t *d2h, *h2d;
  int32_t *step, *ticket, *candidates, *miss_page, *miss_slot, *miss_count, *slot_epoch;
  uint8_t *hit_mask;
};
template <int kLayers>
struct ShortBatch {
  ShortLayer layer[kLayers];
};

constexpr int kShortCopies = 4;   // of a row's histogram
struct alignas(16) ShortShared {
  uint64_t words[kShortRows][kShortList + 4];   // a row's survivors, while it orders them
  uint32_t hist[kShortRows][256 * kShortCopies];
  uint32_t slot_key[kShortSlots];
  uint32_t digit_at[256];
  uint16_t order[2][kShortSlots];               // slots, least recent first, by turns
  uint32_t first[kShortPages];                  // lowest request of a missed page
  int16_t slot_of_page[kShortPages];
  int32_t page_of_slot[kShortSlots];
  uint16_t request[kSelThreads];
  uint16_t victim[kSelThreads], missed[kSelThreads];
  uint32_t touched[kShortSlots / 32];
  uint32_t missed_count[kSelWaves], untouched_count[kSelWaves];
  int32_t step;
  int ordered;                                  // which of the two orders is the result
};

__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
// What other lanes of the wave wrote to LDS ahead of this is read after it.
__device__ __forceinline__ void wave_step() {
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readlane((int)wave_or_to_last_lane(v), 63);
}

// Largest over the wave's lanes (the scan's steps; a lane without a neighbour takes 0).
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
  v = max(v, dpp_u32<0x111, 0xf>(v));
  v = max(v, dpp_u32<0x112, 0xf>(v));
  v = max(v, dpp_u32<0x114, 0xf>(v));
  v = max(v, dpp_u32<0x118, 0xf>(v));
  v = max(v, dpp_u32<0x142, 0xa>(v));
  v = max(v, dpp_u32<0x143, 0xc>(v));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// The k <= kShortList largest of the n <= 64 * kKeys values of `row`, ties by lowest index, in
// order: emit(rank, index).  One wave; `words` and `hist`: its room in LDS.  kLow: the lowest bit
// of a key that says anything (values rounded to a 16-bit type: 16 for bf16, 13 for fp16; key and
// index then fit one word).
template <int kKeys, int kLow, typename Emit>
__device__ __forceinline__ void select_row(const float *row, int n, int k, uint64_t *words, uint32_t *hist,
                                           const Emit &emit) {
  constexpr bool kOneWord = kLow > 0;
  constexpr uint32_t kCounts = ~0u << kLow, kIndex = 0x7ffu;
  static_assert(kKeys * 64 <= kIndex + 1 && (!kOneWord || kIndex < (1u << kLow)), "an index of 11 bits");
  const int lane = threadIdx.x & 63;
  uint32_t key[kKeys];
  uint32_t most = 0, not_least = 0;
  {
    float v[kKeys];
#pragma unroll
    for (int j = 0; j < kKeys; ++j) {
      const int i = j * 64 + lane;
      v[j] = row[i < n ? i : n - 1];
    }
    // (past the end: the smallest key at the highest indices, which displaces no other)
#pragma unroll
    for (int j = 0; j < kKeys; ++j) {
      const uint32_t real = float_order_key(v[j]) & kCounts;
      most = max(most, real);
      not_least = max(not_least, ~real);
      key[j] = j * 64 + lane < n ? real : 0u;
    }
  }
  most = wave_max(most);
  const uint32_t differ = most ^ (~wave_max(not_least) & kCounts);
  // The k-th largest key, eight bits a pass from the highest in which two keys differ: a histogram of the
  // keys that share the bits known so far, a few copies of it, and the bin that holds the k-th.
  int top = differ == 0 ? kLow - 1 : 31 - __builtin_clz(differ);
  uint32_t least = top >= kLow ? most & ~((2u << top) - 1u) : most;
  int want = k;                                  // of the keys that begin like `least`
  bool exact = false;                            // all of those are wanted
  for (bool first = true; top >= kLow && !exact; first = false) {
    const int shift = top - 7 > kLow ? top - 7 : kLow;
    const uint32_t mask = (2u << (top - shift)) - 1u;
#pragma unroll
    for (int u = 0; u < kShortCopies; ++u) *(u32x4 *)(hist + (u * 64 + lane) * 4) = u32x4{0, 0, 0, 0};
    wave_step();
#pragma unroll
    for (int j = 0; j < kKeys; ++j)
      if (first || (key[j] ^ least) >> top < 2u)  // (bits above `top` the same)
        atomicAdd(&hist[(key[j] >> shift & mask) * kShortCopies + (lane & (kShortCopies - 1))], 1u);
    wave_step();
    uint32_t c[4], mine = 0;                     // bins 255 - 4 lane and the three below
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      static_assert(kShortCopies == 4, "a bin's copies are one 16-byte read");
      const u32x4 w = *(const u32x4 *)(hist + (255 - 4 * lane - x) * kShortCopies);
      c[x] = w[0] + w[1] + w[2] + w[3];
      mine += c[x];
    }
    const uint32_t upto = wave_scan_inclusive(mine), before = upto - mine;
    const bool here = before < (uint32_t)want && (uint32_t)want <= upto;     // in one lane
    uint32_t above = before, bin = 255 - 4 * lane, count = c[0];
#pragma unroll
    for (int x = 0; x < 3; ++x)
      if (bin == 255u - 4 * lane - x && above + c[x] < (uint32_t)want) {
        above += c[x];
        count = c[x + 1];
        --bin;
      }
    const int at = __builtin_ctzll(__ballot(here));
    above = (uint32_t)__builtin_amdgcn_readlane((int)above, at);
    bin = (uint32_t)__builtin_amdgcn_readlane((int)bin, at);
    count = (uint32_t)__builtin_amdgcn_readlane((int)count, at);
    least |= bin << shift;
    want -= (int)above;
    exact = want == (int)count;
    top = shift - 1;
  }
  // Compaction, each lane its own: the keys above the threshold (exact: and those that begin like it), in any
  // order; then as many equal to it as are wanted, the lowest indices, by ballots where there are any.
  uint32_t *words32 = (uint32_t *)words;
  auto keep = [&](uint32_t to, int j) {
    const uint32_t i = (uint32_t)(j * 64 + lane);
    if constexpr (kOneWord) words32[to] = key[j] | (kIndex - i);
    else words[to] = (uint64_t)key[j] << 32 | (uint64_t)(kIndex - i);
  };
  auto above_all = [&](auto in) {
    uint32_t mine = 0;
#pragma unroll
    for (int j = 0; j < kKeys; ++j) mine += in(j) ? 1u : 0u;
    uint32_t to = wave_scan_inclusive(mine) - mine;
#pragma unroll
    for (int j = 0; j < kKeys; ++j)
      if (in(j)) keep(to++, j);
  };
  if (exact) {
    above_all([&](int j) { return key[j] >= least && j * 64 + lane < n; });
  } else {
    above_all([&](int j) { return key[j] > least; });
    uint32_t to = (uint32_t)(k - want);
#pragma unroll
    for (int j = 0; j < kKeys; ++j) {
      const uint64_t m = __ballot(key[j] == least);
      if (m == 0 || to >= (uint32_t)k) continue;
      const uint32_t mine = to + lanes_below(m);
      if (key[j] == least && mine < (uint32_t)k) keep(mine, j);
      to += (uint32_t)__popcll(m);
    }
  }
  if (lane < 4) {                                // (zeroes, which beat nothing, up to a whole read)
    if constexpr (kOneWord) words32[k + lane] = 0;
    else words[k + lane] = 0;
  }
  wave_step();
  // Order: all words are distinct, a word's rank is how many are larger.
  auto order = [&](auto two) {
    constexpr int kMine = decltype(two)::value;
    uint32_t rank[kMine] = {}, index[kMine];
    if constexpr (kOneWord) {
      uint32_t mine[kMine];
#pragma unroll
      for (int e = 0; e < kMine; ++e) {
        mine[e] = lane + 64 * e < k ? words32[lane + 64 * e] : 0xffffffffu;
        index[e] = kIndex - (mine[e] & kIndex);
      }
#pragma unroll 4
      for (int i = 0; i < k; i += 4) {
        const u32x4 w = *(const u32x4 *)(words32 + i);
#pragma unroll
        for (int e = 0; e < kMine; ++e)
          rank[e] += (w[0] > mine[e]) + (w[1] > mine[e]) + (w[2] > mine[e]) + (w[3] > mine[e]);
      }
    } else {
      uint64_t mine[kMine];
#pragma unroll
      for (int e = 0; e < kMine; ++e) {
        mine[e] = lane + 64 * e < k ? words[lane + 64 * e] : ~0ull;
        index[e] = kIndex - (uint32_t)mine[e];
      }
#pragma unroll 4
      for (int i = 0; i < k; i += 2) {
        const u64x2 w = *(const u64x2 *)(words + i);
#pragma unroll
        for (int e = 0; e < kMine; ++e) rank[e] += (w[0] > mine[e]) + (w[1] > mine[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < kMine; ++e)
      if (lane + 64 * e < k) emit(rank[e], index[e]);
  };
  if (k <= 64) order(std::integral_constant<int, 1>{});
  else order(std::integral_constant<int, 2>{});
}

// All slots in eviction order (access time, then slot) into sm.order[sm.ordered].  One wave: a
// stable radix sort from the lowest bits in which two times differ up, 8 bits a pass (the times of
// a run lie within few steps: one pass or two).  A pass goes through the slots in their present
// order, 64 at a time: eight ballots say which lanes share a digit, a counter per digit what came before.
__device__ __forceinline__ void order_slots(const float *time, int n_slots, ShortShared &sm) {
  const int lane = threadIdx.x & 63;
  uint32_t ones = 0, zeroes = 0;
  {
    float v[kShortSlotRegs];
#pragma unroll
    for (int j = 0; j < kShortSlotRegs; ++j) {
      const int i = j * 64 + lane;
      v[j] = j * 64 < n_slots ? time[i < n_slots ? i : n_slots - 1] : 0.f;
    }
    // (step counts: as whole numbers they differ in fewer, lower bits than as floats)
    bool whole = true;
#pragma unroll
    for (int j = 0; j < kShortSlotRegs; ++j) whole = whole && v[j] >= 0.f && v[j] <= 0x1p24f && v[j] == truncf(v[j]);
    whole = __all(whole);
#pragma unroll
    for (int j = 0; j < kShortSlotRegs; ++j) {
      const int i = j * 64 + lane;
      if (i < n_slots) {
        const uint32_t key = whole ? (uint32_t)v[j] : float_order_key(v[j]);
        sm.slot_key[i] = key;
        sm.order[0][i] = (uint16_t)i;
        ones |= key;
        zeroes |= ~key;
      }
    }
  }
  uint32_t differ = wave_or(ones) & wave_or(zeroes);
  int from = 0;
  while (differ != 0) {
    const int shift = __builtin_ctz(differ);
    differ &= shift < 24 ? ~0u << (shift + 8) : 0u;
    *(uint4 *)(sm.digit_at + 4 * lane) = make_uint4(0, 0, 0, 0);
    wave_step();
    uint32_t word[kShortSlotRegs];               // slot | place among its digit's << 10 | digit << 20
#pragma unroll
    for (int j = 0; j < kShortSlotRegs; ++j) {
      if (j * 64 < n_slots) {
        const bool valid = j * 64 + lane < n_slots;
        const uint32_t slot = valid ? sm.order[from][j * 64 + lane] : 0u;
        const uint32_t digit = (sm.slot_key[slot] >> shift) & 255u;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          const bool bit = (digit >> b) & 1u;
          const uint64_t with = __ballot(bit);
          peers &= bit ? with : ~with;
        }
        const uint32_t below = lanes_below(peers);
        // (every peer reads the counter before the lowest of them raises it)
        const uint32_t seen = sm.digit_at[digit];
        wave_step();
        if (valid && below == 0) sm.digit_at[digit] = seen + (uint32_t)__popcll(peers);
        wave_step();
        word[j] = slot | (seen + below) << 10 | digit << 20;
      }
    }
    const uint4 c = *(const uint4 *)(sm.digit_at + 4 * lane);
    const uint32_t sum = c.x + c.y + c.z + c.w;
    const uint32_t at = wave_scan_inclusive(sum) - sum;
    wave_step();
    *(uint4 *)(sm.digit_at + 4 * lane) = make_uint4(at, at + c.x, at + c.x + c.y, at + c.x + c.y + c.z);
    wave_step();
#pragma unroll
    for (int j = 0; j < kShortSlotRegs; ++j)
      if (j * 64 + lane < n_slots)
        sm.order[from ^ 1][sm.digit_at[word[j] >> 20] + (word[j] >> 10 & 1023u)] = (uint16_t)(word[j] & 1023u);
    wave_step();
    from ^= 1;
  }
  if (lane == 0) sm.ordered = from;
}

template <int kKeys, int kLow, int kLayers>
__global__ void __launch_bounds__(kSelThreads)
select_update_short_kernel(const ShortBatch<kLayers> batch) {
  __shared__ ShortShared sm;
  const ShortLayer &l = batch.layer[kLayers > 1 ? blockIdx.y : 0];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int h = blockIdx.x, n_heads = gridDim.x;
  const int n_pages = l.n_pages, n_slots = l.n_slots, kp = l.kp, K = l.n_rows * kp;
  float *time = l.time + (int64_t)h * n_slots;
  int64_t *d2h = l.d2h + (int64_t)h * n_pages, *h2d = l.h2d + (int64_t)h * n_slots;

  // both maps into LDS, by the waves that have nothing else to do
  const int busy = l.n_rows, idle = kSlotWave - busy;     // waves [busy, kSlotWave)
  if (wave >= busy && wave < kSlotWave) {
    const int first = (wave - busy) * 64 + lane, stride = idle * 64;
#pragma unroll 4
    for (int i = first; i < n_pages; i += stride) {
      sm.slot_of_page[i] = (int16_t)d2h[i];
      sm.first[i] = 0xffffffffu;
    }
#pragma unroll 2
    for (int i = first; i < n_slots; i += stride) sm.page_of_slot[i] = (int32_t)h2d[i];
    for (int i = first; i < kShortSlots / 32; i += stride) sm.touched[i] = 0;
    if (first == 0) sm.step = *l.step;
  } else if (wave == kSlotWave) {
    order_slots(time, n_slots, sm);
  } else {
    const float *row = l.scores + ((int64_t)wave * n_heads + h) * n_pages;
    int64_t *dst = l.idx + (int64_t)h * K + wave * kp;
    uint16_t *request = sm.request + wave * kp;
    select_row<kKeys, kLow>(row, n_pages, kp, sm.words[wave], sm.hist[wave], [=](uint32_t rank, uint32_t page) {
      dst[rank] = (int64_t)page;
      request[rank] = (uint16_t)page;
    });
  }
  __syncthreads();

  // The last head to have read the step counter publishes its new value and re-arms the ticket.
  const int32_t step = sm.step + 1;
  const float now = (float)step;
  if (t == 0) {
    if (atomicAdd(l.ticket, 1) == n_heads - 1) {
      *l.step = step;
      *l.ticket = 0;
    }
  }
  // hits are touched, the first request of every missed page is found
  int page = -1, slot = -1;
  if (t < K) {
    page = sm.request[t];
    slot = sm.slot_of_page[page];
    if (slot >= 0) {
      time[slot] = now;
      atomicOr(&sm.touched[slot >> 5], 1u << (slot & 31));
    } else {
      atomicMin(&sm.first[page], (uint32_t)t);
    }
  }
  const uint16_t *order = sm.order[sm.ordered];
  const int old_slot = t < n_slots ? order[t] : -1;
  if (t < l.k_cand) l.candidates[(int64_t)h * l.k_cand + t] = old_slot;
  if (t == 0) l.candidates[(int64_t)n_heads * l.k_cand + h] = step - 1;   // (the step the list describes)
  __syncthreads();
  // the i-th missed page, in the order of the requests, takes the i-th least recent slot that no
  // request touched (K <= n_slots: there are enough)
  const bool miss = t < K && slot < 0 && sm.first[page] == (uint32_t)t;
  const bool untouched = old_slot >= 0 && !(sm.touched[old_slot >> 5] >> (old_slot & 31) & 1u);
  if (t < K && l.hit_mask) l.hit_mask[(int64_t)h * K + t] = miss ? 0 : 1;
  const uint64_t m_miss = __ballot(miss), m_untouched = __ballot(untouched);
  if (lane == 0) {
    sm.missed_count[wave] = (uint32_t)__popcll(m_miss);
    sm.untouched_count[wave] = (uint32_t)__popcll(m_untouched);
  }
  __syncthreads();
  uint32_t n_miss, n_untouched;
  const uint32_t miss_at = waves_prefix(sm.missed_count, n_miss) + lanes_below(m_miss);
  const uint32_t untouched_at = waves_prefix(sm.untouched_count, n_untouched) + lanes_below(m_untouched);
  if (miss) sm.missed[miss_at] = (uint16_t)page;
  if (untouched) sm.victim[untouched_at] = (uint16_t)old_slot;
  __syncthreads();
  if (t < (int)n_miss) {
    const int p = sm.missed[t], v = sm.victim[t], old = sm.page_of_slot[v];
    if (old >= 0 && old < n_pages) d2h[old] = -1;
    h2d[v] = p;
    d2h[p] = v;
    time[v] = now;
    l.miss_page[(int64_t)h * K + t] = p;
    l.miss_slot[(int64_t)h * K + t] = v;
    if (l.slot_epoch) l.slot_epoch[(int64_t)h * n_slots + v] = step;
  }
  if (t == 0) l.miss_count[h] = (int32_t)n_miss;
}

bool topk_lru_short(const da_decode_step_args &a) {
  const int rep = a.n_q_heads / a.n_kv_heads;
  return a.n_pages <= kShortPages && rep <= kShortRows && a.kp <= kShortList && rep * a.kp <= kSelThreads &&
         a.n_slots <= (a.n_pages <= 1024 ? kShortSlots : 896) && rep * a.kp <= a.n_slots;
}

template <int kKeys, int kLow, int kLayers>
static void launch_short(const da_decode_step_args *a, int n, hipStream_t s) {
  ShortBatch<kLayers> batch;
  for (int i = 0; i < n; ++i)
    batch.layer[i] = {a[i].scores, a[i].n_q_heads / a[i].n_kv_heads, (int)a[i].n_pages, a[i].kp, a[i].n_slots,
                      a[i].k_cand, a[i].idx, a[i].access_time, a[i].d2h, a[i].h2d, a[i].step,
                      (int32_t *)a[i].lru_workspace, a[i].candidates, a[i].miss_page, a[i].miss_slot, a[i].miss_count,
                      a[i].slot_epoch, a[i].hit_mask};
  hipLaunchKernelGGL((select_update_short_kernel<kKeys, kLow, kLayers>), dim3(a->n_kv_heads, n),
                     dim3(kSelThreads), 0, s, batch);
}

template <int kKeys, int kLow>
static void launch_short(const da_decode_step_args *a, int n, hipStream_t s) {
  if (n == 1) launch_short<kKeys, kLow, 1>(a, n, s);
  else launch_short<kKeys, kLow, kStepBatch>(a, n, s);
}

template <int kLow>
static void launch_short(const da_decode_step_args *a, int n, hipStream_t s) {
  if (a->n_pages <= 512) launch_short<8, kLow>(a, n, s);
  else if (a->n_pages <= 1024) launch_short<16, kLow>(a, n, s);
  else launch_short<32, kLow>(a, n, s);
}

int launch_topk_lru_short(const da_decode_step_args *a, int n, hipStream_t s) {
  bool rounded = a->dtype != DA_F32;      // (layers may differ in their flags)
  for (int i = 0; i < n; ++i) rounded = rounded && (a[i].score_flags & DA_SCORE_ROUND);
  if (!rounded) launch_short<0>(a, n, s);
  else if (a->dtype == DA_BF16) launch_short<16>(a, n, s);
  else launch_short<13>(a, n, s);
  return launch_status("da_decode_step(selection of short rows)");
}

}  // namespace da
