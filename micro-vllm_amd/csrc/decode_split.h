// The split-KV decode tile loop of the pipelined decode kernel, as a device
// function: the decode kernel (attention_decode.hip) and the one-launch
// attention step (attention_prefill.hip), which runs decode and prefill
// workgroups in one grid, both call it.
//
// Work item: (KV head, split of the visible context, request). One wavefront
// owns one KV head; a workgroup holds `waves` consecutive KV heads of the
// same (request, split), so together they stream whole token rows (all heads
// of a token are contiguous in the cache). Per 16-token tile a wave computes
// S^T = K . Q^T with v_mfma_f32_16x16x32 (M = 16 tokens, N = the G query heads
// of the KV head, padded to 16, K = head_dim: 64, 96 or 128); the softmax runs
// on the accumulator layout, and P^T is the B operand of O^T += V^T . P^T
// (v_mfma_f32_16x16x16), fed as a hi/lo pair so the product keeps ~16 mantissa
// bits (more at head_dim 64 and 96: kSplitParts); the V^T operand comes from
// transposing LDS reads (ds_read_b64_tr_b16).
#pragma once

#include <cmath>
#include <type_traits>

#include "worklists.h"

namespace mvllm {
namespace {
namespace dec {

template <typename T>
__device__ __forceinline__ void split_hi_lo(float p, uint32_t& hi, uint32_t& lo) {
  hi = Elem<T>::to_bits(p);
  lo = Elem<T>::to_bits(p - Elem<T>::from_bits(hi));
}

// ---------------------------------------------------------------------------
// Partials of a request with several splits, and their merge.
//
// The workgroup that finishes a request's last open split merges the partials
// in the same launch. Workgroups of one request run on different XCDs, whose
// L2 caches are not coherent with each other, so the partials are written and
// read past them (sc1: agent-scope stores and loads, the same bits that
// relaxed agent-scope atomics carry): each workgroup's stores are complete
// (vmcnt 0) before it counts itself done, and the one that counts last reads
// only after that. No cache-wide write-back or invalidation is involved (with
// a device-scope fence per workgroup the 256-sequence Qwen3 batch's kernel had
// taken 590 us instead of 372). A merge kernel of its own cost 4-9 us per
// forward: the launch, then two or three dependent rounds of loads.

typedef uint32_t uint4_ext __attribute__((ext_vector_type(4)));
constexpr int kAgentScope = 16;  // sc1 in a buffer instruction's cache-policy operand

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_at(void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(base, 0, -1, 0x00020000);
}

// Merges `ns` partials (rows base, base + 1, ...) of query token `qs` for `heads`
// query heads from `head0`, one wave: 32 lanes per query head, 4 dims each
// (at head_dim 64 and 96 the last lanes only merge statistics), with the
// log-sum-exp rule. A round takes up to CAP splits (MANY: several rounds) of
// PAIRS pairs of heads, about 32 rows, whose loads are issued together.
template <typename T, int D, int CAP, bool MANY>
__device__ __forceinline__ void merge_splits(const AttnArgs& a, int64_t base, int64_t qs, int head0, int heads, int ns) {
  static_assert(CAP <= 32, "one lane per split of a round");
  constexpr int PAIRS = CAP <= 8 ? 4 : CAP <= 16 ? 2 : 1;
  const int sub = threadIdx.x & 31;
  const int half = (threadIdx.x >> 5) & 1;
  const bool has_dims = 4 * sub < D;
  const int d0 = has_dims ? 4 * sub : 0;
  const int64_t row0 = base * a.num_q_heads;  // partial row of (split 0, head 0)
  for (int g0 = 0; g0 < heads; g0 += 2 * PAIRS) {
    auto pair_live = [&](int p) { return g0 + 2 * p < heads; };  // wave-uniform
    auto head_live = [&](int p) { return g0 + 2 * p + half < heads; };
    auto head = [&](int p) { return head0 + g0 + 2 * p + (head_live(p) ? half : 0); };
    // This lane's split of a round: its (max, sum), or (-inf, 0) past the end.
    auto round_stats = [&](int s0, int p) {
      const bool own = sub < CAP && s0 + sub < ns;
      int s = own ? s0 + sub : 0;
      asm volatile("" : "+v"(s));  // one load for all lanes, not one per side of the condition
      const uint64_t w = __hip_atomic_load(
          reinterpret_cast<const uint64_t*>(a.ws_ml) + row0 + head(p) + static_cast<int64_t>(s) * a.num_q_heads,
          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return own ? make_float2(__uint_as_float(static_cast<uint32_t>(w)), __uint_as_float(static_cast<uint32_t>(w >> 32)))
                 : make_float2(-INFINITY, 0.f);
    };
    float mx[PAIRS], sum[PAIRS];
    float4_t o[PAIRS];
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
      mx[p] = -INFINITY;
      sum[p] = 0.f;
      o[p] = float4_t{0.f, 0.f, 0.f, 0.f};
      if constexpr (MANY) {
        for (int s0 = CAP; s0 < ns; s0 += CAP) mx[p] = fmaxf(mx[p], round_stats(s0, p).x);
      }
    }
    for (int s0 = 0; s0 < (MANY ? ns : 1); s0 += CAP) {
      float2 ml[PAIRS];
      float4_t v[PAIRS][CAP];
      const __amdgpu_buffer_rsrc_t rows = buffer_at(a.ws_acc + (row0 + static_cast<int64_t>(s0) * a.num_q_heads) * D);
#pragma unroll
      for (int p = 0; p < PAIRS; ++p) {
        if (!pair_live(p)) continue;
        ml[p] = round_stats(s0, p);
#pragma unroll
        for (int j = 0; j < CAP; ++j) {
          const int k = s0 + j < ns ? j : ns - 1 - s0;  // past the last split: re-read, unused
          v[p][j] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                     rows, 4 * ((k * a.num_q_heads + head(p)) * D + d0), 0, kAgentScope));
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // every load before the first use
#pragma unroll
      for (int p = 0; p < PAIRS; ++p) {
        if (!pair_live(p)) continue;
        if (s0 == 0) {
          mx[p] = fmaxf(mx[p], ml[p].x);
#pragma unroll
          for (int m = 16; m >= 1; m >>= 1) mx[p] = fmaxf(mx[p], __shfl_xor(mx[p], m, 32));
        }
        // A split with no visible key (m = -inf) weighs 0; so does every split
        // when none has one, and the output is then NaN (0 / 0).
        const float w = ml[p].x == -INFINITY ? 0.f : exp2f(ml[p].x - mx[p]);
        sum[p] += w * ml[p].y;
#pragma unroll
        for (int j = 0; j < CAP; ++j) {
          const float wj = __shfl(w, j, 32);
          if (s0 + j < ns) o[p] += v[p][j] * wj;
        }
      }
    }
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
      if (!pair_live(p)) continue;
#pragma unroll
      for (int m = 16; m >= 1; m >>= 1) sum[p] += __shfl_xor(sum[p], m, 32);
      const float inv = 1.f / sum[p];
      if (head_live(p) && has_dims) {
        uint16_t* op = static_cast<uint16_t*>(a.out) + qs * a.o_s0 + static_cast<int64_t>(head(p)) * a.o_s1;
        *reinterpret_cast<uint2*>(op + d0) =
            uint2{Elem<T>::to_bits(o[p][0] * inv) | (Elem<T>::to_bits(o[p][1] * inv) << 16),
                  Elem<T>::to_bits(o[p][2] * inv) | (Elem<T>::to_bits(o[p][3] * inv) << 16)};
      }
    }
  }
}

// merge_splits with the round that fits `ns`.
template <typename T, int D>
__device__ __forceinline__ void merge_request(const AttnArgs& a, int64_t base, int64_t qs, int head0, int heads, int ns) {
  if (ns <= 2) merge_splits<T, D, 2, false>(a, base, qs, head0, heads, ns);
  else if (ns <= 4) merge_splits<T, D, 4, false>(a, base, qs, head0, heads, ns);
  else if (ns <= 8) merge_splits<T, D, 8, false>(a, base, qs, head0, heads, ns);
  else if (ns <= 16) merge_splits<T, D, 16, false>(a, base, qs, head0, heads, ns);
  else if (ns <= 24) merge_splits<T, D, 24, false>(a, base, qs, head0, heads, ns);
  else if (ns <= 32) merge_splits<T, D, 32, false>(a, base, qs, head0, heads, ns);
  else merge_splits<T, D, 32, true>(a, base, qs, head0, heads, ns);
}

// Epilogue shared by the decode kernels, entered by every wave of the
// workgroup (`live`: the wave has a KV head). acc[b][e] is
// O[head h*G + col][dim 16b + 4grp + e] (unnormalised), m / lt the running
// max (exp2 domain) and the complete softmax denominator of this split. A
// request with one split gets its output directly; otherwise the partial goes
// to the workspace, and the workgroup that completes the request (for its
// group of KV heads, `head_group`) merges the partials. `flag`: an LDS word
// that no wave uses any more once all have entered. MERGE false: a launch of its
// own merges every batch (the merge's registers are not needed).
template <typename T, int D, bool MERGE>
__device__ __forceinline__ void finish_split(const AttnArgs& a, const DecodeItem& item, int h, bool live, int head_group,
                                             int head_groups, float m, float lt, const float4_t (&acc)[D / 16],
                                             int32_t* flag) {
  const int col = threadIdx.x & 15;
  const int grp = (threadIdx.x >> 4) & 3;
  const int G = a.group;
  if (item.ns == 1) {
    if (!live || col >= G) return;
    const float inv = 1.f / lt;
    uint16_t* op = static_cast<uint16_t*>(a.out) + item.qs * a.o_s0 + static_cast<int64_t>(h * G + col) * a.o_s1;
#pragma unroll
    for (int b = 0; b < D / 16; ++b) {
      const uint32_t w0 = Elem<T>::to_bits(acc[b][0] * inv) | (Elem<T>::to_bits(acc[b][1] * inv) << 16);
      const uint32_t w1 = Elem<T>::to_bits(acc[b][2] * inv) | (Elem<T>::to_bits(acc[b][3] * inv) << 16);
      *reinterpret_cast<uint2*>(op + 16 * b + 4 * grp) = uint2{w0, w1};
    }
    return;
  }
  if (live && col < G) {
    // Partial row of (this split, head h * G); the lanes' heads follow it.
    const int64_t row = (static_cast<int64_t>(item.base) + item.split) * a.num_q_heads +
                        static_cast<int64_t>(__builtin_amdgcn_readfirstlane(h)) * G;
    const __amdgpu_buffer_rsrc_t rows = buffer_at(a.ws_acc + row * D);
#pragma unroll
    for (int b = 0; b < D / 16; ++b)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4_ext, acc[b]), rows, 4 * (col * D + 16 * b + 4 * grp), 0,
                                             kAgentScope);
    if (grp == 0)
      __hip_atomic_store(reinterpret_cast<uint64_t*>(a.ws_ml) + row + col,
                         static_cast<uint64_t>(__float_as_uint(m)) | (static_cast<uint64_t>(__float_as_uint(lt)) << 32),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if constexpr (MERGE) {
    if (a.merge_apart) return;
    // This wave's partials have reached the point all XCDs read from.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int32_t* const counter = a.done + static_cast<int64_t>(item.r) * head_groups + head_group;
    if (threadIdx.x == 0) {
      // Counts to ns and wraps to zero for the next launch, in one operation: a
      // reset of its own would lose counts that another launch on this workspace
      // added in between, and leave the counter off for every later one.
      const uint32_t last = static_cast<uint32_t>(item.ns) - 1;
      *flag = atomicInc(reinterpret_cast<unsigned int*>(counter), last) == last;
    }
    __syncthreads();
    if (!*flag || !live) return;
    merge_request<T, D>(a, item.base, item.qs, __builtin_amdgcn_readfirstlane(h) * G, G, item.ns);
  }
}

// Output rows that no split writes, kTidyTokens tokens and as many requests
// per workgroup `wg`: zeros for tokens outside every request (the reference's
// zeros_like output), and NaN for a decode request with no visible key
// (softmax over no keys) and, in a batch whose hint promised single-query
// requests only, for the rows of any other request, which no kernel computes.
constexpr int kTidyTokens = 16;

inline int64_t tidy_blocks(const AttnArgs& a) {
  const int64_t most = a.num_tokens > a.num_requests ? a.num_tokens : a.num_requests;
  return (most + kTidyTokens - 1) / kTidyTokens;
}

template <typename T>
__device__ inline void tidy_rows(const AttnArgs& a, int64_t wg) {
  const int64_t R = a.num_requests;
  const int64_t first = a.qsl[0], last = a.qsl[R];
  // Rows are contiguous (16-byte aligned, head_dim a multiple of 8).
  auto fill_row = [&](int64_t t, uint32_t bits2) {
    uint16_t* op = static_cast<uint16_t*>(a.out) + t * a.o_s0;
    const int chunks = a.head_dim / 8;
    for (int i = threadIdx.x; i < a.num_q_heads * chunks; i += blockDim.x) {
      const int hq = i / chunks, c = i - hq * chunks;
      *reinterpret_cast<uint4*>(op + hq * a.o_s1 + 8 * c) = uint4{bits2, bits2, bits2, bits2};
    }
  };
  const int64_t t0 = wg * kTidyTokens;
  if (t0 < first || t0 + kTidyTokens > last) {
    for (int64_t t = t0; t < t0 + kTidyTokens && t < a.num_tokens; ++t)
      if (t < first || t >= last) fill_row(t, 0u);
  }
  const uint32_t nan_bits = Elem<T>::to_bits(NAN);
  const uint32_t nan2 = nan_bits | (nan_bits << 16);
  for (int64_t r = t0; r < t0 + kTidyTokens && r < R; ++r) {
    const int2 req = a.decode_req[r];  // (query token, splits; -1: not a decode request)
    if (req.y == 0 && req.x >= 0 && req.x < a.num_tokens) fill_row(req.x, nan2);
    if (req.y >= 0 || !a.decode_only) continue;
    const int64_t q0 = a.qsl[r], q1 = a.qsl[r + 1];
    if (q0 < 0 || q1 > a.num_tokens) continue;
    for (int64_t t = q0; t < q1; ++t) fill_row(t, nan2);
  }
}

// ---------------------------------------------------------------------------
// Pipelined variant for block sizes that are multiples of 16 (every 16-token
// tile then lies in one block). K and V tiles go straight from HBM to LDS
// (global_load_lds_dwordx4): each load instruction covers 1 KiB of whole rows
// (4 tokens of 256 B at head_dim 128, 8 of 128 B at 64), i.e. whole 128-byte
// lines, except at head_dim 96 whose 192-byte rows share them. tile_phys gives
// the 16-byte chunk of a row in which a tile's logical chunk lies; it is a
// permutation within the row, so the lanes of a load stay inside the same
// lines on the global side, and it spreads both LDS read patterns over the
// banks: the K rows as MFMA A operands (16 rows, one chunk) and the
// transposing V reads (8 rows, two neighbouring chunks). STAGES tiles per wave
// are in flight; waits are explicit vmcnt counts because the only
// vector-memory instructions in the loop are these tile loads (the split's
// block ids are fetched once, up front).
//
// A lone wave's tile took 2,650 cycles when the loads of tile k + 1 were issued
// from 64-bit lane addresses before tile k was read (issue 820, S 465, softmax
// 440, P.V 800 behind its LDS reads); scalar load addresses, the tile read to
// registers first and the refill issued behind those reads shorten it, and
// keep a tile more in flight where HBM is the bound. The loads carry the non-temporal
// hint: every K/V byte is read exactly once, and keeping the stream from
// displacing other cached lines raised the measured bandwidth from 5.5 to
// 6.0 TB/s on the Qwen3 decode batch.

// P^T enters P.V in 16-bit parts. At head_dim 128: a hi/lo pair. At 64 and 96
// requests have always been answered with fp32 probabilities, which three parts
// of bf16 hold whole (256 decodes of 2,000 keys: 186 us, 185 with a pair); two of
// fp16 hold 22 bits, down to 2^-29 of the maximum, with P lifted by 2^15 and the
// second part by another 2^11 and summed apart, out of the subnormals.
template <typename T, int D>
constexpr int kSplitParts = D != 128 && std::is_same_v<T, bf16_t> ? 3 : 2;
template <typename T, int D>
constexpr bool kSumLow = D != 128 && !std::is_same_v<T, bf16_t>;
constexpr float kLift = 32768.f, kLowScale = 2048.f;

template <int D> constexpr int kTileBytesOf = 16 * 2 * D;  // one 16-token tile of one head, K or V

// Tiles in flight per wave: 32 KiB of K and V per wave for the narrow heads
// too, whose tiles are smaller (two workgroups of four waves share a CU's LDS).
template <int D> constexpr int kStages = D == 64 ? 4 : D == 96 ? 3 : 2;

// Physical 16-byte chunk of logical chunk q in row t (t < 16) of a tile.
// D = 128 (16 chunks, one bank row): XOR with t rotated left by one bit.
// D = 64 (8 chunks, two rows per bank row): XOR with the bit-reversed t / 2.
// D = 96 (12 chunks; row starts fall on four bank offsets): rotated by t / 4.
template <int D>
__device__ __forceinline__ int tile_phys(int t, int q) {
  if constexpr (D == 128) {
    return q ^ (((t << 1) | (t >> 3)) & 15);
  } else if constexpr (D == 64) {
    const int u = (t >> 1) & 7;
    return q ^ (((u & 1) << 2) | (u & 2) | (u >> 2));
  } else {
    const int x = q + (t >> 2);
    return x >= 12 ? x - 12 : x;
  }
}

// The logical chunk held by physical chunk p of row t.
template <int D>
__device__ __forceinline__ int tile_logical(int t, int p) {
  if constexpr (D == 96) {
    const int x = p - (t >> 2);
    return x < 0 ? x + 12 : x;
  } else {
    return tile_phys<D>(t, p);  // an XOR is its own inverse
  }
}

// Waits until at most `tiles` tiles of LOADS loads each are outstanding
// (wave-uniform, at most 3).
template <int LOADS>
__device__ __forceinline__ void wait_tiles(int tiles) {
  if (tiles >= 3) wait_vmcnt<3 * LOADS>();
  else if (tiles == 2) wait_vmcnt<2 * LOADS>();
  else if (tiles == 1) wait_vmcnt<LOADS>();
  else wait_vmcnt<0>();
}

typedef short tr_short4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) tr_short4 lds_tr_short4;
typedef __attribute__((address_space(3))) const short8_t lds_short8;

template <typename T, int D, int STAGES>
__device__ __forceinline__ void decode_split_lds_body(const AttnArgs& a, uint8_t* smem, uint32_t wg, int waves) {
  constexpr int kTileBytes = kTileBytesOf<D>;
  constexpr int kLoads = D / 32;  // 1 KiB loads per K (or V) tile
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int col = lane & 15;
  const int grp = lane >> 4;
  // 1-D grid: workgroup b takes head group b % groups of work-list slot b / groups.
  const int groups = (a.num_kv_heads + waves - 1) / waves;
  const int h = static_cast<int>(wg % groups) * waves + wave;
  // The work-list record carries the request's query token, visible range
  // and this split's key range, so the first tile loads wait on two
  // dependent loads (the record, then the block ids) rather than four.
  const int64_t slot = wg / groups;
  if (slot >= a.item_capacity) {  // past the work list's capacity
    tidy_rows<T>(a, static_cast<int64_t>(wg) - a.item_capacity * groups);
    return;
  }
  const DecodeItem item = a.decode_items[slot];
  if (item.r < 0 || item.r >= a.num_requests) return;
  const bool live = h < a.num_kv_heads;  // a spare wave only joins the epilogue's barriers
  const int split = item.split;
  const int64_t r = item.r;
  const int64_t qs = item.qs;
  const int64_t lo = item.lo;
  const int64_t begin = item.begin;
  const int64_t end = item.end;
  // Records index the query, the table and the partials: out-of-range
  // fields (never written by the work-list kernel) end the workgroup.
  if (begin < 0 || begin > end || end - begin >= a.split_tokens || end >= a.width * a.block_size ||
      qs < 0 || qs >= a.num_tokens || split < 0 || split >= item.ns || item.base < 0 ||
      static_cast<int64_t>(item.base) + item.ns > a.item_capacity)
    return;
  const int ntiles = live ? static_cast<int>((end - begin) / 16 + 1) : 0;  // <= 128 (split <= 2048)

  // Block id and in-block row of tiles `lane` and `lane + 64` of this split,
  // fetched once (block ids are < 2^31; a 16-aligned tile never straddles a
  // block).
  int32_t my_block[2] = {-1, -1}, my_row[2] = {0, 0};
  if (a.page_shift >= 0) {
    // A power-of-two number of 16-token pages per block: shifts instead of
    // 64-bit divisions.
    const int64_t* const table_row = a.table + r * a.t_s0;
    int64_t id[2] = {-1, -1};
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const uint32_t page = (static_cast<uint32_t>(begin) >> 4) + lane + 64 * x;
      my_row[x] = static_cast<int32_t>((page & ((1u << a.page_shift) - 1u)) << 4);
      if (lane + 64 * x < ntiles) id[x] = table_row[static_cast<int64_t>(page >> a.page_shift) * a.t_s1];
    }
#pragma unroll
    for (int x = 0; x < 2; ++x) my_block[x] = id[x] >= 0 && id[x] < a.num_blocks ? static_cast<int32_t>(id[x]) : -1;
  } else {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      if (lane + 64 * x < ntiles) {
        const int64_t p = begin + 16 * (lane + 64 * x);
        my_block[x] = static_cast<int32_t>(block_of(a, r, p));
        my_row[x] = static_cast<int32_t>(p % a.block_size);
      }
    }
  }
  // Tile t's block id and row (t wave-uniform).
  auto tile_block = [&](int t) {
    return t < 64 ? __builtin_amdgcn_readlane(my_block[0], t) : __builtin_amdgcn_readlane(my_block[1], t - 64);
  };
  auto tile_row = [&](int t) {
    return t < 64 ? __builtin_amdgcn_readlane(my_row[0], t) : __builtin_amdgcn_readlane(my_row[1], t - 64);
  };

  const int G = a.group;
  const int hq = h * G + col;
  short8_t qv[kLoads];
  {
    const uint16_t* qp = static_cast<const uint16_t*>(a.q) + qs * a.q_s0 +
                         static_cast<int64_t>(live && col < G ? hq : 0) * a.q_s1 + 8 * grp;
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      qv[i] = (live && col < G) ? *reinterpret_cast<const short8_t*>(qp + 32 * i) : short8_t{0, 0, 0, 0, 0, 0, 0, 0};
  }

  uint8_t* wave_lds = smem + static_cast<size_t>(wave) * STAGES * 2 * kTileBytes;
  const uint32_t wave_lds_addr = __builtin_amdgcn_readfirstlane(lds_address(wave_lds));
  const uint16_t* cache = static_cast<const uint16_t*>(a.cache);
  const int64_t head_elems = static_cast<int64_t>(h) * D;

  // Load-side mapping: instruction i, this lane -> 16-byte chunk 64i + lane of
  // the tile's LDS slot (byte offset of its data from the tile's first row;
  // decode_supported's callers keep 16 rows within 32 bits).
  uint32_t lane_off[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int t = (64 * i + lane) / (D / 8);
    const int p = (64 * i + lane) % (D / 8);
    lane_off[i] = static_cast<uint32_t>(2 * (t * a.c_s[2] + 8 * tile_logical<D>(t, p)));
  }
  // Read-side byte offsets within a tile: K row `col`, chunk 4i + grp; and the
  // transposing V reads, in which lane 4k + c of a 16-lane group points at row
  // 4grp + k, dims 16b + 4c .. +4.
  int koff[kLoads], voff[D / 16];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) koff[i] = 2 * D * col + 16 * tile_phys<D>(col, 4 * i + grp);
#pragma unroll
  for (int b = 0; b < D / 16; ++b) {
    const int t = 4 * grp + (col >> 2);
    voff[b] = 2 * D * t + 16 * tile_phys<D>(t, 2 * b + ((col & 3) >> 1)) + 8 * (col & 1);
  }

  auto issue = [&](int tile, int stage) {
    const int32_t blk = tile_block(tile);
    const int32_t row = tile_row(tile);
    const uint32_t dst = wave_lds_addr + stage * 2 * kTileBytes;
    // An invalid block id masks the whole tile: block 0 is read instead.
    const int64_t at = blk >= 0 ? static_cast<int64_t>(blk) * a.c_s[1] + static_cast<int64_t>(row) * a.c_s[2] : 0;
    const uint16_t* const tile_k = cache + at + head_elems;
    const uint16_t* const tile_v = tile_k + a.c_s[0];
    lds_dma_load16_stream<0>(tile_k, lane_off[0], dst);
    lds_dma_load16_stream<kTileBytes>(tile_v, lane_off[0], dst);
    lds_dma_load16_stream<1024>(tile_k, lane_off[1], dst);
    lds_dma_load16_stream<kTileBytes + 1024>(tile_v, lane_off[1], dst);
    if constexpr (kLoads > 2) {
      lds_dma_load16_stream<2048>(tile_k, lane_off[2], dst);
      lds_dma_load16_stream<kTileBytes + 2048>(tile_v, lane_off[2], dst);
    }
    if constexpr (kLoads > 3) {
      lds_dma_load16_stream<3072>(tile_k, lane_off[3], dst);
      lds_dma_load16_stream<kTileBytes + 3072>(tile_v, lane_off[3], dst);
    }
  };

  constexpr int kParts = kSplitParts<T, D>;
  constexpr bool kLow = kSumLow<T, D>;
  float4_t acc[D / 16];
  float m, l;
  // One walk over the split's tiles; EXACT: with P in fp32
  // (v_mfma_f32_16x16x4_f32; as the only walk it took 31.1 us instead of 24.6 for
  // 8 decodes of 4,000 keys at head_dim 96 and 2 KV heads).
  auto walk = [&](auto exact_c) {
    constexpr bool EXACT = decltype(exact_c)::value;
    float4_t low[D / 16];  // kLow: the product with the second parts
#pragma unroll
    for (int b = 0; b < D / 16; ++b) acc[b] = low[b] = float4_t{0.f, 0.f, 0.f, 0.f};
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
      if (s < ntiles) issue(s, s);

    for (int k = 0; k < ntiles; ++k) {
      const int stage = k % STAGES;
      const int later = (ntiles - 1 - k) < (STAGES - 1) ? (ntiles - 1 - k) : (STAGES - 1);
      wait_tiles<2 * kLoads>(later);
      __builtin_amdgcn_wave_barrier();
      compiler_fence();

      // The whole tile goes to registers first, so that its stage refills while
      // it is computed (STAGES tiles in flight throughout) and the V reads do
      // not wait behind the softmax.
      const uint32_t kt = wave_lds_addr + stage * 2 * kTileBytes;
      const uint32_t vt = kt + kTileBytes;
      short8_t kf[kLoads];
      uint2 vf[D / 16];
#pragma unroll
      for (int i = 0; i < kLoads; ++i)
        kf[i] = *reinterpret_cast<lds_short8*>(static_cast<uintptr_t>(kt + koff[i]));
#pragma unroll
      for (int b = 0; b < D / 16; ++b) {
        // A operand: lane (col, grp) receives V[token 4grp + e][dim 16b + col].
        vf[b] = __builtin_bit_cast(
            uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_tr_short4*>(static_cast<uintptr_t>(vt + voff[b]))));
      }
      // All LDS reads of this stage retire before the refill is issued.
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      compiler_fence();
      __builtin_amdgcn_sched_barrier(0);
      if (k + STAGES < ntiles) issue(k + STAGES, stage);

      const int32_t tb = static_cast<int32_t>(begin) + 16 * k;
      // Token j of the tile is visible iff its position is in [lo, end] and the block is valid.
      uint32_t okmask = 0;
      if (tile_block(k) >= 0) {
        const int32_t first_ok = lo > tb ? static_cast<int32_t>(lo) - tb : 0;
        const int32_t last_ok = end - tb < 15 ? static_cast<int32_t>(end) - tb : 15;
        okmask = (last_ok >= first_ok) ? ((0xFFFFu >> (15 - last_ok)) & (0xFFFFu << first_ok)) : 0u;
      }

      float4_t sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < kLoads; ++i) sc = Mfma<T>::k32(kf[i], qv[i], sc);
      float s[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        s[e] = ((okmask >> (4 * grp + e)) & 1u) ? sc[e] * a.scale_log2 : -INFINITY;
      float bm = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
      bm = max_xor32_f(max_xor16_f(bm));
      const float mn = fmaxf(m, bm);
      // v_exp_f32 flushes results below 2^-126 to zero: nothing beside the
      // row's maximum of 1.
      const float alpha = (mn == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f(m - mn);
      float p[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) p[e] = (s[e] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(s[e] - mn);
      l = l * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
      if (__ballot(alpha != 1.f)) {
#pragma unroll
        for (int b = 0; b < D / 16; ++b) {
          acc[b] *= alpha;
          if constexpr (kLow && !EXACT) low[b] *= alpha;
        }
      }
      m = mn;

      if (okmask != 0xFFFFu) {
        // Rows of masked tokens may hold stale or non-finite data: zero them in V.
        const uint32_t ok4 = okmask >> (4 * grp);
        const uint32_t mlo = (ok4 & 1u ? 0xFFFFu : 0u) | (ok4 & 2u ? 0xFFFF0000u : 0u);
        const uint32_t mhi = (ok4 & 4u ? 0xFFFFu : 0u) | (ok4 & 8u ? 0xFFFF0000u : 0u);
#pragma unroll
        for (int b = 0; b < D / 16; ++b) vf[b] = uint2{vf[b].x & mlo, vf[b].y & mhi};
      }
      if constexpr (!EXACT) {
        short4_t part[kParts];
        float rest[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) rest[e] = kLow ? p[e] * kLift : p[e];
#pragma unroll
        for (int y = 0; y < kParts; ++y) {
          uint32_t w[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            w[e] = Elem<T>::to_bits(rest[e]);
            rest[e] -= Elem<T>::from_bits(w[e]);
            if constexpr (kLow) rest[e] *= kLowScale;
          }
          part[y] = __builtin_bit_cast(short4_t, uint2{w[0] | (w[1] << 16), w[2] | (w[3] << 16)});
        }
        // The products of a block depend on each other, the blocks do not.
#pragma unroll
        for (int y = 0; y < kParts; ++y)
#pragma unroll
          for (int b = 0; b < D / 16; ++b) {
            float4_t& to = kLow && y == 1 ? low[b] : acc[b];
            to = Mfma<T>::k16(__builtin_bit_cast(short4_t, vf[b]), part[y], to);
          }
      } else {
        // Step x: k index grp stands for token 4grp + x, whose probability and V
        // row the lane holds already.
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int b = 0; b < D / 16; ++b) {
            const uint32_t w = x < 2 ? vf[b].x : vf[b].y;
            acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(Elem<T>::from_bits(x & 1 ? w >> 16 : w & 0xFFFFu), p[x], acc[b],
                                                          0, 0, 0);
          }
      }
    }
    if constexpr (kLow && !EXACT) {
#pragma unroll
      for (int b = 0; b < D / 16; ++b) acc[b] = (acc[b] + low[b] * (1.f / kLowScale)) * (1.f / kLift);
    }
  };
  // The block ids and Q must be in registers before the first tile address.
  __builtin_amdgcn_s_waitcnt(0);
  walk(std::false_type{});
  // At head_dim 64 and 96 an infinity in V stays one, as in the any-shape kernel:
  // times a part of P that is zero or negative it is NaN, which no later tile
  // takes out of the accumulators again. Such a wave answers its split with P in
  // fp32.
  if constexpr (D != 128) {
    float zero = 0.f;
#pragma unroll
    for (int b = 0; b < D / 16; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) zero = __builtin_fmaf(acc[b][e], 0.f, zero);
    if (__ballot(zero != zero)) walk(std::true_type{});
  }

  const float lt = sum_xor32_f(sum_xor16_f(l));
  // The flag lies in the first wave's K tile: written after every wave's loop.
  finish_split<T, D, true>(a, item, h, live, static_cast<int>(wg % groups), groups, m, lt, acc, reinterpret_cast<int32_t*>(smem));
}

}  // namespace dec
}  // namespace
}  // namespace mvllm
