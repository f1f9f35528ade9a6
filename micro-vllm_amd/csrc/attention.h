// Internal interface shared by the attention kernels.
#pragma once

#include "common.h"

namespace mvllm {

// One decode work-list record: split `split` (of `ns`) of request `r`, whose
// single query is token `qs` with visible keys from `lo`; the split streams
// keys [begin, end], and its partial goes to row `base` + `split` of the
// partials. Positions fit in int32 (the launcher checks the block table's
// reach). r = -1 marks an empty slot.
struct DecodeItem {
  int32_t r, split, qs, ns;
  int32_t lo, base, begin, end;
};

// Longest split that the pipelined decode kernel takes: it reads a split's
// block ids once, two 16-token tiles per lane. (The general kernel, which has
// no such limit, streams ~15% slower: 1,097 against 916 us on 64 contexts of
// 8k-33k tokens.)
constexpr int32_t kMaxSplit = 2048;

// One prefill work-list record: query tokens [t0, t1) of request `r` (whose
// first query is token `qs`); lo is the first visible key of row t0 and hi
// the last visible key of row t1 - 1 (their hull covers every row when
// visible ranges grow with the token, which the kernel checks). r = -1
// marks an empty slot.
struct PrefillItem {
  int32_t r, t0, t1, qs;
  int32_t lo, hi, pad0, pad1;
};

// How long the decode splits are (worklists.h): rates in split tokens per token
// of the batch, and bounds.
struct SplitRule {
  float small, full;                // while the work does not fill the chip; when it does
  float beside_small, beside_full;  // the same beside prefill work
  float waves;                      // one wave per SIMD
  float fits;                       // 1 / (slots beyond one per request), or 0
  float whole;                      // longest request answered whole, per token of the batch
  int32_t whole_decodes;            // requests that fill the chip by themselves
  int32_t least;                    // a shorter split than this is only for few tokens
  int32_t shortest;                 // no split is shorter
  int32_t beside_most;              // longest split beside prefill work
  int32_t merge_apart;              // the partials are merged by a launch of their own
  int32_t beside_merge;             // splits per request beside prefill work, up to 128 tokens each (0: no bound)
};

// Everything a ragged paged-attention launch needs. Strides are in elements.
struct AttnArgs {
  const void* q;
  int64_t q_s0, q_s1, q_s2;
  const void* cache;
  int64_t c_s[5];
  void* out;
  int64_t o_s0, o_s1, o_s2;
  const int64_t* positions;
  const int64_t* cstarts;
  const int64_t* qsl;
  const int64_t* lengths;
  const int64_t* table;
  int64_t t_s0, t_s1, width;
  int64_t num_tokens, num_requests, num_blocks, block_size;
  int32_t num_q_heads, num_kv_heads, group, head_dim;
  float scale_log2;  // softmax scale * log2(e): scores live in the exp2 domain
  // log2(block_size / 16) when block_size is a multiple of 16 whose
  // quotient is a power of two (16-key pages are then found with shifts),
  // else -1.
  int32_t page_shift = -1;
  // Split-KV decode partials: acc [item_capacity][Hq][D], (max, sum)
  // [item_capacity][Hq]; a request's splits take consecutive rows.
  float* ws_acc;
  float2* ws_ml;
  int64_t item_capacity;  // slots of the decode work list
  int32_t split_tokens;   // bound on the length of a split
  int32_t split_fixed;    // the length of every split, or 0: chosen with the work list
  int32_t num_cus;
  SplitRule rule;
  int32_t mode;  // generic kernel: 0 = every token; 1 = only requests with > 1 query
  // Prefill work list: one record per (request, query block) slot, heaviest
  // first; r = -1 marks an empty slot. Written by the item kernel before the
  // prefill kernel reads it.
  PrefillItem* items;
  // Decode work list: one record per (request, split), full splits first, then
  // the partial last splits from the largest; r = -1 marks an empty slot.
  DecodeItem* decode_items;
  // Per request, written with the decode work list: (query token, number of
  // splits), or (0, -1) for a request that is not a single-query decode. The
  // rows that no split writes are found from it.
  int2* decode_req;
  // Per (request, group of KV heads that share a workgroup): splits finished
  // so far in this launch. Zeroed with the work list; the count wraps to zero
  // with the workgroup that completes a request.
  int32_t* done;
  // The partials are merged by a launch of their own (merge_apart in
  // attention_api.hip); `done` then holds each request's first partial row.
  int32_t merge_apart;
  // Host side only: the work lists and the per-request table are already in
  // the workspace (planned once for a step), so the launches skip the
  // work-list kernels.
  int32_t lists_ready;
  // The caller's max_query_len hint said 1 (no prefill launch): the rows of
  // any request with another query count are made NaN (tidy_rows).
  int32_t decode_only;
};

// Visible key positions [lo, hi] of query `t` in request `r` whose first
// query is `qs`: the reference gathers [start(first query), length) and
// masks keys outside [start(t), pos(t)] (reference.py:101-138, 49-68).
// Positions past the block table's reach cannot be mapped and are clipped.
__device__ __forceinline__ void visible_range(const AttnArgs& a, int64_t r, int64_t qs,
                                              int64_t t, int64_t& lo, int64_t& hi) {
  const int64_t first = a.cstarts[qs];
  const int64_t own = a.cstarts[t];
  lo = own > first ? own : first;
  if (lo < 0) lo = 0;
  hi = a.positions[t];
  const int64_t last = a.lengths[r] - 1;
  if (last < hi) hi = last;
  const int64_t reach = a.width * a.block_size - 1;
  if (reach < hi) hi = reach;
}

// Physical block holding position p of request r, or -1 when the table
// entry is not a valid block id (such keys are treated as masked).
__device__ __forceinline__ int64_t block_of(const AttnArgs& a, int64_t r, int64_t p) {
  const int64_t b = a.table[r * a.t_s0 + (p / a.block_size) * a.t_s1];
  return (b >= 0 && b < a.num_blocks) ? b : -1;
}

// Host-side launchers (one per kernel family).
// Launchers; `start`/`stop` (may be null) bracket the main kernel's launch.
int launch_generic(const AttnArgs& a, int32_t dtype, hipStream_t s);
int launch_decode(const AttnArgs& a, int32_t dtype, hipStream_t s, hipEvent_t start,
                  hipEvent_t stop);
// The decode partials' merge, where it is a launch of its own (launch_decode
// includes it).
int launch_merge(const AttnArgs& a, int32_t dtype, hipStream_t s);
// The work-list kernels alone (decode list + per-request table; prefill list).
int launch_decode_lists(const AttnArgs& a, hipStream_t s);
int launch_prefill_lists(const AttnArgs& a, hipStream_t s);
int launch_prefill(const AttnArgs& a, int32_t dtype, hipStream_t s, hipEvent_t start,
                   hipEvent_t stop);
bool prefill_supported(const AttnArgs& a, int32_t dtype);

// The one-launch attention step: decode and prefill workgroups in one grid
// (attention_prefill.hip), for batches whose decode part runs the pipelined
// kernel with its default shape (kStepDecodeWaves waves; two stages at head_dim
// 128, three at 96, four at 64).
constexpr int kStepDecodeWaves = 4;
bool decode_step_eligible(const AttnArgs& a);
// The split-KV decode kernels cover this head_dim with this block size and
// split length (128 always; 64 and 96 with the pipelined kernel only).
bool decode_supported(int64_t head_dim, int64_t block_size, int64_t split_tokens);
// 16 rows of this stride lie within a 32-bit byte offset, as the pipelined
// decode kernel addresses them (the general one, at head_dim 128, does not).
inline bool rows_within_32_bits(int64_t token_stride) { return 32 * token_stride < (int64_t{1} << 32); }
// The batch's decodes run on the general split kernel.
bool decode_general(const AttnArgs& a);
int64_t decode_step_blocks(const AttnArgs& a);  // decode workgroups of the step grid
// `prefill_first`: the prefill workgroups lead the grid (else the decode ones).
int launch_step(const AttnArgs& a, int32_t dtype, bool prefill_first, hipStream_t s, hipEvent_t start,
                hipEvent_t stop);

// Device properties used for launch shapes (cached per device).
int device_cu_count();

}  // namespace mvllm
