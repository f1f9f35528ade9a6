// Work-list builders of the attention kernels and the KV-row copy, as
// device functions: each runs in one 1024-thread workgroup (the list
// builders) or a part of one (the row copy), either in its own kernel or in
// the fused prologue of a forward (attention_api.hip), which builds both
// lists and writes the step's K/V rows in a single launch.
#pragma once

#include "attention.h"

namespace mvllm {

// One token's K and V rows copied into its cache slot (bit-exact), 16 bytes
// per step: whole token rows, because all KV heads of one token are
// contiguous in the cache layout (2, blocks, block_size, heads, dim).
struct KvRowArgs {
  const char* key;
  const char* value;
  char* cache;
  const int64_t* slots;
  int64_t key_token_stride;    // bytes
  int64_t value_token_stride;  // bytes
  int64_t plane_stride;        // bytes
  int64_t block_stride;        // bytes
  int64_t offset_stride;       // bytes
  int64_t block_size;
  int64_t num_slots;
  int32_t chunks;              // 16-byte chunks per token row
};

// Validates a KV write (mvllm_kv_write's checks) and, when the rows can be
// copied 16 bytes at a time, fills `rows` and sets `*vectorised` (kv_cache.hip).
int kv_write_prepare(const mvllm_tensor3* key, const mvllm_tensor3* value, const mvllm_kv_cache* cache,
                     const int64_t* slot_mapping, int64_t num_tokens, KvRowArgs* rows, bool* vectorised);

namespace {

// Rows of one prefill workgroup: (query head of a KV head's group, token)
// pairs; a work item then covers T = kRows / G query tokens, and
// prefill_lg_tok gives log2(T).
constexpr int kRows = 128;

inline int prefill_lg_tok(const AttnArgs& a) {
  int lg_tok = 0;
  while ((kRows >> lg_tok) > a.group) ++lg_tok;
  return lg_tok;
}

// Chunks c = first, first + step, ... of token `token`'s K row then V row.
// A slot < 0 or >= num_slots writes nothing.
__device__ inline void copy_kv_row(const KvRowArgs& a, int64_t token, int first, int step) {
  const int64_t slot = a.slots[token];
  const char* ksrc = a.key + token * a.key_token_stride;
  const char* vsrc = a.value + token * a.value_token_stride;
  if (first < 2 * a.chunks && first + step >= 2 * a.chunks) {
    // One chunk per thread: its load does not depend on the slot, so it is
    // issued before the slot is known and the two latencies overlap (a
    // padding token's row exists too; only its store is skipped).
    const bool is_value = first >= a.chunks;
    const int chunk = is_value ? first - a.chunks : first;
    const uint4 data = *reinterpret_cast<const uint4*>((is_value ? vsrc : ksrc) + 16 * chunk);
    // Keep the slot's checks (and their wait) after the load is issued.
    __builtin_amdgcn_sched_barrier(0);
    if (slot < 0 || slot >= a.num_slots) return;
    const int64_t block = slot / a.block_size;
    const int64_t offset = slot - block * a.block_size;
    char* dst = a.cache + block * a.block_stride + offset * a.offset_stride;
    *reinterpret_cast<uint4*>(dst + (is_value ? a.plane_stride : 0) + 16 * chunk) = data;
    return;
  }
  if (slot < 0 || slot >= a.num_slots) return;
  const int64_t block = slot / a.block_size;
  const int64_t offset = slot - block * a.block_size;
  char* dst = a.cache + block * a.block_stride + offset * a.offset_stride;
  for (int c = first; c < 2 * a.chunks; c += step) {
    const bool is_value = c >= a.chunks;
    const int chunk = is_value ? c - a.chunks : c;
    const uint4 data = *reinterpret_cast<const uint4*>((is_value ? vsrc : ksrc) + 16 * chunk);
    *reinterpret_cast<uint4*>(dst + (is_value ? a.plane_stride : 0) + 16 * chunk) = data;
  }
}

// ---- decode work list --------------------------------------------------------
//
// One workgroup lists the (request, split) items of the single-query
// requests: every full split first (in any order), then the partial last
// splits from the largest down, so the in-order dispatch of the decode grid
// ends on the shortest items. Empty slots (up to the capacity) get request -1.
//
// The split length follows from the visible tokens, which only the device
// knows; the numbers of items it aims at follow from the shape (split_rule). A
// split costs a workgroup ~5 us besides its tiles (metadata, the pipeline's
// start, the partial and its merge), and a tile of a workgroup that has a CU to
// itself ~0.65 us. A workgroup holds up to four KV heads, one wave each, so an
// item is ceil(heads / 4) workgroups, of fewer waves below four heads. So (us per
// forward, captured back to back; head_dim 128, narrower tokens count by their
// bytes):
// * while the work does not fill the chip, one workgroup for three quarters of
//   the CUs, of 64 to 256 tokens; with two or three KV heads, whose workgroups
//   leave room, one per CU of up to 192, and with one head two of up to 128. 8
//   contexts of 128 .. 4,096 with 8 heads: 36.1 with 64-token splits, 23.3 with
//   192, 34.1 with 512; one context of 1,024: 13.7 with 64, 21.0 with 256. 96
//   items whatever the heads, as for 8, had taken, for 32 contexts of 500 ..
//   1,000 with 4 heads 23.5 (18.9 with 192 items) and with 2 23.1 (17.3 with
//   256), and for 4 of 1,000 .. 2,000 with 16 heads 23.2 (20.9 with 48);
// * beyond that, about two items per CU of up to 1,024 tokens (64 contexts of
//   8k .. 33k: 868, 907 with 2,048; 256 of 128 .. 4,096: 361, 379 with 256),
//   four with fewer than four KV heads (128 contexts of 2,000 .. 4,000 with 14/2
//   heads: 90 with two per CU, 82 with four);
// * beside prefill work, whose workgroups fill the chip as well, half an item per
//   CU of up to 2,048 (248 decodes and 8 chunks of 512: 736 with 2,048, 781 with
//   512). One per CU of up to 768 with four KV heads (128 decodes of 3,000 ..
//   6,000 and a chunk of 40 with 32/4: 230 with 2,048, 216 with 768), and one and
//   a half per CU below four (128 of 1,000 .. 2,000 with one KV head: 84.5 with
//   half an item per CU, 39 with one and a half);
// * no splits at all where the requests alone fill the chip (workgroups for
//   three quarters of the CUs), are about even or short, and the longest one's
//   tiles take no longer than the whole batch takes at the HBM's rate (0.04 us
//   per token against ~6.2 TB/s): the partials and their merge are then pure
//   cost. 201 decodes that see 484 keys each: 70 us whole, 77-81 in two or
//   three splits; 256 of 505: 85.5 and 93; 128 of 20 .. 300: 23.0 and 26.1
//   (uneven ones of up to 965 keys are better off split: 83.0 whole, 80.6);
// * at most 32 splits per request up to 512 tokens each: the merge loads 32
//   at a time (one context of 32k: 143 us with 64-token splits, 47 with 512).
//   Where a launch of its own merges, a wave per two heads: 32 up to 256, then 64
//   while the work leaves SIMDs idle (one context of 16k with 28/4 heads: 39.6
//   with 512, 33.0 with 256; four with 32/8: 49 with 512, 57 with 256). Beside
//   prefill work 16 up to 128 tokens each where one wave merges more than four
//   heads (a context of 2,000 and a chunk of 40 with 32/4 heads: 25.8 with 64,
//   22.2 with 128).
// The general split kernel (block sizes that are not multiples of 16) keeps four
// waves per SIMD and waits longer for each tile: two items per CU of 64 to 1,024
// tokens whatever the heads, and no requests left whole (17 contexts of up to 1,670
// with 10 heads in blocks of 8: 46.8 by the rule above, 34.6 so).
// At least total / (capacity - R), so that the items fit the list: a request
// of v tokens has at most v / split + 1 splits. (2,048-token splits always fit:
// see item_slots.)
constexpr int kDecodeListThreads = 1024;
constexpr int kSizeBuckets = 64;  // sizes of a partial split, split / 64 tokens (rounded up to a power of two) each
constexpr int32_t kSmallSplit = 64, kMostSplit = 1024;
constexpr int32_t kGeneralWhole = 128;  // reach up to which the general split kernel answers requests whole

// Items (of 128-wide tokens) that a batch is split into, at most, by the rule above.
inline int32_t small_items(int32_t cus, int32_t num_kv_heads) {
  const int32_t items =
      num_kv_heads == 1 ? 2 * cus : num_kv_heads < 4 ? cus : 3 * cus / (4 * ((num_kv_heads + 3) / 4));
  return items > 1 ? items : 1;
}
inline int32_t full_items(int32_t cus, int32_t num_kv_heads) { return num_kv_heads < 4 ? 4 * cus : 2 * cus; }
inline int32_t full_split(int32_t num_kv_heads) { return num_kv_heads == 1 ? 128 : num_kv_heads < 4 ? 192 : 256; }

// The general split kernel leaves its merge to a launch, which a batch without
// splits does not need: up to 128 tokens one wave answers a request about as fast
// as two and the merge (a context of 102 with 16/1 heads in blocks of 8: 15.0 us,
// 16.3 split; 229 of up to 78 with 48/8 22.8, 26.5 with the launch), of 160 not (8
// with 16/8 heads: 21.6, 18.5).
inline bool general_merges(int64_t reach, int64_t split_fixed) { return split_fixed || reach > kGeneralWhole; }

// The rule's numbers for a shape. Rates turn tokens into a split length.
// `general`: the general split kernel runs.
inline SplitRule split_rule(const AttnArgs& a, bool general) {
  const int32_t heads = a.num_kv_heads, cus = a.num_cus;
  const float width = a.head_dim / 128.f;
  SplitRule r;
  r.small = width / small_items(cus, heads);
  r.full = width / full_items(cus, heads);
  r.beside_small = width / 96.f;
  r.beside_full = width / (heads < 4 ? 1.5f * cus : heads == 4 ? 1.f * cus : 0.5f * cus);
  r.waves = width * heads / (4.f * cus);
  r.fits = a.item_capacity > a.num_requests ? 1.f / static_cast<float>(a.item_capacity - a.num_requests) : 0.f;
  r.whole = heads * a.head_dim / (0.04f * 1.55e6f);
  r.whole_decodes = (3 * cus + 4 * ((heads + 3) / 4) - 1) / (4 * ((heads + 3) / 4));
  r.least = full_split(heads);
  r.shortest = kSmallSplit;
  r.beside_most = heads == 4 ? 768 : kMaxSplit;
  r.merge_apart = a.merge_apart;
  r.beside_merge = !a.merge_apart && a.group > 4 ? 16 : 0;
  if (general) {
    r.small = r.full = r.beside_small = r.beside_full = width / (2.f * cus);
    // Without the merge launch (general_merges) no request may be split.
    r.least = r.shortest = a.merge_apart ? kSmallSplit : kGeneralWhole;
    r.whole_decodes = INT32_MAX;
    r.beside_most = kMostSplit;
  }
  return r;
}

// Slots of the decode work list and of the decode grid, from shapes alone: at
// most `capacity` (the workspace's) and no more than choose_split can fill. A
// slot that stays empty still costs a workgroup's dispatch (~4 ns, 6 us for
// 1,500 of them).
// Splits of 2,048 tokens fit every one of the bounds.
// `decodes`: the batch looks like decodes alone. Beside prefill work spare slots
// cost more than their dispatch: the work is then spread over the CUs unevenly (8
// decodes of 2,000 and a chunk of 500 with 32/4 heads: 27.5, 32.0 with 96 more).
inline int64_t item_slots(int64_t requests, int64_t reach, int64_t capacity, int64_t cus, int64_t head_dim,
                          int32_t num_kv_heads, bool decodes, bool general) {
  auto least = [](int64_t x, int64_t y) { return x < y ? x : y; };
  auto larger = [](int64_t x, int64_t y) { return x > y ? x : y; };
  const int64_t tokens = requests * reach;
  const int64_t small = (decodes ? small_items(static_cast<int32_t>(cus), num_kv_heads) : 96) * 128 / head_dim + 1;
  const int64_t full = least(full_items(static_cast<int32_t>(cus), num_kv_heads) * 128LL / head_dim,
                             tokens / full_split(num_kv_heads)) + 1;
  const int64_t any = least(2 * cus * 128 / head_dim, tokens / kSmallSplit) + 1;
  const int64_t slots = requests + larger(general ? any : larger(small, full), tokens / kMostSplit + 1);
  return least(least(slots, requests * ((reach + kSmallSplit - 1) / kSmallSplit)), capacity);
}

__host__ __device__ inline int32_t choose_split(int64_t total, int32_t longest, int32_t decodes, bool beside_prefill,
                                       const SplitRule& rule) {
  // Quotients as products in float (divisions take longer than the rest of the
  // rule), raised by more than their error; lengths past 2^20 mean the same.
  auto up16 = [](float v) { return (static_cast<int32_t>(fminf(v * 1.000001f, 1048576.f)) + 16) & ~15; };
  const float tokens = static_cast<float>(total);
  if (!beside_prefill && longest <= kMostSplit && decodes >= rule.whole_decodes &&
      (longest <= 320 || tokens >= 0.75f * longest * decodes) && longest <= tokens * rule.whole)
    return (longest + 15) & ~15;
  const int32_t most = beside_prefill ? rule.beside_most : kMostSplit;
  int32_t split = up16(tokens * (beside_prefill ? rule.beside_full : rule.full));
  int32_t least = up16(tokens * (beside_prefill ? rule.beside_small : rule.small));
  least = least < rule.shortest ? rule.shortest : least > rule.least ? rule.least : least;
  if (beside_prefill && rule.beside_merge > 0) {
    const int32_t few = longest / rule.beside_merge < 112 ? (longest / rule.beside_merge + 16) & ~15 : 128;
    least = least < few ? few : least;
  }
  split = split < least ? least : split > most ? most : split;
  int32_t by_merge = (longest / 32 + 16) & ~15;
  if (rule.merge_apart && by_merge > 256) {
    const int32_t by_waves = up16(tokens * rule.waves);
    const int32_t by_64 = (longest / 64 + 16) & ~15;
    const int32_t more = by_64 > by_waves ? by_64 : by_waves;
    by_merge = more < 256 ? 256 : more < by_merge ? more : by_merge;
  }
  if (split < by_merge) split = by_merge < 512 ? by_merge : split < 512 ? 512 : split;
  const int32_t fits = rule.fits > 0.f ? up16(tokens * rule.fits) : kMaxSplit;
  if (split < fits) split = fits;
  return split < kMaxSplit ? split : kMaxSplit;
}

__device__ inline void build_decode_list(const AttnArgs& a) {
  __shared__ int32_t full_count, full_pos, base_pos, longest, others, decodes;
  __shared__ unsigned long long pages;
  __shared__ int32_t bucket[kSizeBuckets];
  const int tid = threadIdx.x;
  const int64_t R = a.num_requests;
  const int64_t capacity = a.item_capacity;
  if (tid == 0) {
    full_count = full_pos = base_pos = longest = others = decodes = 0;
    pages = 0;
  }
  if (tid < kSizeBuckets) bucket[tid] = 0;
  // A decode request: its query token, visible keys and their number from the
  // 16-aligned position below the first (0: none, or not a decode request;
  // dec = 1 marks a decode request).
  struct Desc {
    int32_t qs, lo, hi, tokens, dec;
  };
  const Desc none = {0, 0, -1, 0, 0};
  auto describe = [&](int64_t r) {
    Desc d = none;
    const int64_t qs = a.qsl[r];
    if (qs < 0 || qs >= a.num_tokens || a.qsl[r + 1] - qs != 1) return d;
    d.qs = static_cast<int32_t>(qs);
    d.dec = 1;
    int64_t lo, hi;
    visible_range(a, r, qs, qs, lo, hi);
    if (hi < lo) return d;
    d.lo = static_cast<int32_t>(lo);
    d.hi = static_cast<int32_t>(hi);
    d.tokens = static_cast<int32_t>(hi - (lo & ~int64_t(15)) + 1);
    return d;
  };
  // The thread's first request stays in registers between the passes.
  const Desc d0 = tid < R ? describe(tid) : none;
  auto desc_of = [&](int64_t r) { return r >= R ? none : r == tid ? d0 : describe(r); };
  __syncthreads();
  const int lane = tid & 63;
  // Exclusive prefix of v over the wave and the wave's total.
  auto wave_scan = [&](int32_t v, int32_t& sum) {
    int32_t incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t y = __shfl_up(incl, d, 64);
      if (lane >= d) incl += y;
    }
    sum = __shfl(incl, 63, 64);
    return incl - v;
  };
  // Pass 0: visible 16-token pages in all, the longest range, and whether any
  // request is not a decode. The loop bounds are uniform per wave. A wave sums
  // the low 16 bits of its page counts and the rest apart, so neither
  // overflows.
  const auto add = [](int32_t x, int32_t y) { return x + y; };
  const auto larger = [](int32_t x, int32_t y) { return x > y ? x : y; };
  int32_t split = a.split_fixed;
  if (split == 0) {
    for (int64_t r0 = tid - lane; r0 < R; r0 += kDecodeListThreads) {
      const Desc d = desc_of(r0 + lane);
      const int32_t count = (d.tokens >> 4) + ((d.tokens & 15) != 0);
      const int32_t low = wave_reduce_i(count & 0xFFFF, add);
      const int32_t high = wave_reduce_i(count >> 16, add);
      const int32_t most = wave_reduce_i(d.tokens, larger);
      const bool other = __ballot(r0 + lane < R && !d.dec) != 0;
      const int32_t seen = static_cast<int32_t>(__popcll(__ballot(d.tokens > 0)));
      if (lane == 0) {
        atomicAdd(&pages, (static_cast<unsigned long long>(high) << 16) + low);
        atomicMax(&longest, most);
        if (other) others = 1;
        atomicAdd(&decodes, seen);
      }
    }
    __syncthreads();
    split = choose_split(16 * static_cast<int64_t>(pages), longest, decodes, others && !a.decode_only, a.rule);
  }
  // 64 buckets of 2^bucket_shift sizes span every split length: the smallest
  // shift with 64 << shift >= split (a partial split holds 1 .. split - 1
  // keys, so its bucket index stays below 64).
  const int bucket_shift = split <= kSizeBuckets ? 0 : 32 - __builtin_clz((split - 1) / kSizeBuckets);
  auto splits_of = [&](const Desc& d) { return (d.tokens + split - 1) / split; };
  // Pass 1: count full splits (one LDS atomic per wave), histogram the
  // partial ones by size.
  for (int64_t r0 = tid - lane; r0 < R; r0 += kDecodeListThreads) {
    const Desc d = desc_of(r0 + lane);
    const int32_t ns = splits_of(d);
    const int32_t last = d.tokens - (ns - 1) * split;
    const bool partial = ns > 0 && last < split;
    const int32_t sum = wave_reduce_i(partial ? ns - 1 : ns, add);
    if (lane == 0 && sum) atomicAdd(&full_count, sum);
    if (partial) atomicAdd(&bucket[(last - 1) >> bucket_shift], 1);
  }
  __syncthreads();
  // Partial splits start after the full ones, largest bucket first: an
  // exclusive scan over the buckets in descending order, one lane each.
  static_assert(kSizeBuckets == 64, "one wave scans the buckets");
  if (tid < 64) {
    const int32_t c = bucket[63 - tid];
    int32_t sum;
    const int32_t excl = wave_scan(c, sum);
    const int32_t fulls = full_count;
    bucket[63 - tid] = fulls + excl;
    if (tid == 63) full_count = fulls + sum;  // total number of items
  }
  __syncthreads();
  // Pass 2: place the items (one LDS atomic per wave for the full splits and
  // one for the requests' partial rows).
  for (int64_t r0 = tid - lane; r0 < R; r0 += kDecodeListThreads) {
    const int64_t r = r0 + lane;
    const Desc d = desc_of(r);
    const int32_t ns = splits_of(d);
    const int32_t last = d.tokens - (ns - 1) * split;
    const bool partial = ns > 0 && last < split;
    const int32_t nfull = partial ? ns - 1 : ns;
    int32_t rows;
    const int32_t row_excl = wave_scan(ns, rows);
    const uint64_t partials = __ballot(partial);
    const int32_t before = __popcll(partials & ((uint64_t{1} << lane) - 1));  // partial splits of lower lanes
    int32_t at = 0, base = 0;
    if (lane == 0 && rows) {
      at = atomicAdd(&full_pos, rows - static_cast<int32_t>(__popcll(partials)));
      base = atomicAdd(&base_pos, rows);
    }
    at = __builtin_amdgcn_readfirstlane(at) + row_excl - before;
    base = __builtin_amdgcn_readfirstlane(base) + row_excl;
    auto place = [&](int32_t slot, int32_t sp) {
      const int32_t begin = (d.lo & ~15) + sp * split;
      const int32_t end = begin + split - 1 < d.hi ? begin + split - 1 : d.hi;
      if (slot < capacity) a.decode_items[slot] = DecodeItem{static_cast<int32_t>(r), sp, d.qs, ns, d.lo, base, begin, end};
    };
    for (int32_t sp = 0; sp < nfull; ++sp) place(at + sp, sp);
    if (partial) place(atomicAdd(&bucket[(last - 1) >> bucket_shift], 1), ns - 1);
    if (r < R) {
      a.decode_req[r] = int2{d.qs, d.dec ? ns : -1};
      if (a.merge_apart) a.done[r] = base;
    }
  }
  // At most one counter per (request, KV head).
  if (!a.merge_apart)
    for (int64_t j = tid; j < R * a.num_kv_heads; j += kDecodeListThreads) a.done[j] = 0;
  for (int64_t j = full_count + tid; j < capacity; j += kDecodeListThreads)
    a.decode_items[j] = DecodeItem{-1, -1, 0, 0, 0, 0, 0, -1};
}


// ---- prefill work list ------------------------------------------------------
//
// Request r's query blocks of T tokens occupy work-list slots
// [qsl[r] / T + r, qsl[r] / T + r + ceil(n_r / T)), which never overlap and
// stay below N / T + R. One workgroup lists every (request, block) item of
// the multi-query requests, sorted by the number of 64-key tiles it visits,
// heaviest first, so that the hardware's in-order dispatch of the prefill
// grid approximates longest-processing-time-first scheduling. Empty slots
// (single-query requests) go last as request -1. Items within a cost
// bucket come in any order; every item writes only its own output rows.
constexpr int kItemThreads = 1024;
constexpr int kItemSlots = 8192;    // larger batches keep slot order (late slots first)
constexpr int kCostBuckets = 2048;  // tiles per item, clamped
static_assert(kCostBuckets == 2 * kItemThreads, "the bucket scan gives each thread two buckets");

__device__ inline void build_prefill_list(const AttnArgs& a, int32_t lg_tok) {
  __shared__ int32_t owner[kItemSlots];
  __shared__ uint16_t bucket_of[kItemSlots];
  __shared__ int32_t start[kCostBuckets];
  __shared__ int32_t wave_sums[kItemThreads / 64];
  __shared__ int32_t total;
  const int tid = threadIdx.x;
  const int64_t tpb = int64_t{1} << lg_tok;
  const int64_t R = a.num_requests;
  const int64_t nslots = a.num_tokens / tpb + R;
  // Record of query block b of request r (its first query is qs, its last
  // query token qe - 1).
  auto record = [&](int64_t r, int64_t qs, int64_t qe, int64_t b) {
    const int64_t t0 = qs + b * tpb;
    const int64_t t1 = t0 + tpb < qe ? t0 + tpb : qe;
    int64_t lo0, hi0, lo1, hi1;
    visible_range(a, r, qs, t0, lo0, hi0);
    visible_range(a, r, qs, t1 - 1, lo1, hi1);
    return PrefillItem{static_cast<int32_t>(r), static_cast<int32_t>(t0), static_cast<int32_t>(t1),
                       static_cast<int32_t>(qs), static_cast<int32_t>(lo0), static_cast<int32_t>(hi1), 0, 0};
  };
  const PrefillItem empty = {-1, 0, 0, 0, 0, -1, 0, 0};
  if (nslots > kItemSlots) {
    for (int64_t j = tid; j < nslots; j += kItemThreads) {
      int64_t rl = 0, rh = R - 1;
      while (rl < rh) {
        const int64_t mid = (rl + rh + 1) >> 1;
        if (a.qsl[mid] / tpb + mid <= j) rl = mid; else rh = mid - 1;
      }
      const int64_t qs = a.qsl[rl], qe = a.qsl[rl + 1];
      const int64_t b = j - (qs / tpb + rl);
      const bool ok = qs >= 0 && qe <= a.num_tokens && qe - qs > 1 && b >= 0 && qs + b * tpb < qe;
      a.items[nslots - 1 - j] = ok ? record(rl, qs, qe, b) : empty;
    }
    return;
  }
  for (int j = tid; j < nslots; j += kItemThreads) owner[j] = -1;
  for (int k = tid; k < kCostBuckets; k += kItemThreads) start[k] = 0;
  __syncthreads();
  for (int64_t r = tid; r < R; r += kItemThreads) {
    const int64_t qs = a.qsl[r], qe = a.qsl[r + 1];
    if (qs < 0 || qe > a.num_tokens || qe - qs <= 1) continue;
    const int64_t first = qs / tpb + r;
    const int64_t nb = (qe - qs + tpb - 1) / tpb;
    for (int64_t b = 0; b < nb && first + b < nslots; ++b) owner[first + b] = static_cast<int32_t>(r);
  }
  __syncthreads();
  // Cost of an item: 64-key tiles between its first row's first visible key
  // and its last row's last one.
  for (int j = tid; j < nslots; j += kItemThreads) {
    const int32_t r = owner[j];
    if (r < 0) continue;
    const int64_t qs = a.qsl[r], qe = a.qsl[r + 1];
    const int64_t t0 = qs + (j - (qs / tpb + r)) * tpb;
    const int64_t t1 = (t0 + tpb < qe ? t0 + tpb : qe) - 1;
    int64_t lo0, hi0, lo1, hi1;
    visible_range(a, r, qs, t0, lo0, hi0);
    visible_range(a, r, qs, t1, lo1, hi1);
    const int64_t tiles = hi1 >= lo0 ? (hi1 - lo0 + 64) / 64 : 0;
    const int bucket = static_cast<int>(tiles < kCostBuckets - 1 ? tiles : kCostBuckets - 1);
    bucket_of[j] = static_cast<uint16_t>(bucket);
    atomicAdd(&start[bucket], 1);
  }
  __syncthreads();
  // start[k] = number of items in buckets above k (exclusive scan, heaviest
  // first). Thread t owns buckets K - 1 - 2 t and K - 2 - 2 t.
  {
    const int k0 = kCostBuckets - 1 - 2 * tid;
    const int v0 = start[k0], v1 = start[k0 - 1];
    const int own = v0 + v1;
    int incl = own;
    const int lane = tid & 63, w = tid >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(incl, d, 64);
      if (lane >= d) incl += y;
    }
    if (lane == 63) wave_sums[w] = incl;
    __syncthreads();
    int before = 0;
    for (int i = 0; i < w; ++i) before += wave_sums[i];
    const int excl = before + incl - own;
    if (tid == kItemThreads - 1) total = excl + own;
    __syncthreads();
    start[k0] = excl;
    start[k0 - 1] = excl + v0;
  }
  __syncthreads();
  for (int j = tid; j < nslots; j += kItemThreads) {
    const int32_t r = owner[j];
    if (r < 0) continue;
    const int pos = atomicAdd(&start[bucket_of[j]], 1);
    const int64_t qs = a.qsl[r], qe = a.qsl[r + 1];
    a.items[pos] = record(r, qs, qe, j - (qs / tpb + r));
  }
  for (int64_t j = total + tid; j < nslots; j += kItemThreads) a.items[j] = empty;
}


}  // namespace
}  // namespace mvllm
