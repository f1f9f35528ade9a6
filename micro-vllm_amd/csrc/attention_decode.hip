// Split-KV ragged decode on gfx950 matrix cores (bf16/fp16; head_dim 128, and
// 64 and 96 where the block size is a multiple of 16).
//
// Work item: (KV head, split of the visible context, request). One wavefront
// owns one KV head; a workgroup holds up to 8 waves = 8 consecutive KV heads
// of the same (request, split), so together they stream whole token rows
// (all heads of a token are contiguous in the cache) with 16-byte loads.
// A one-workgroup kernel lists the (request, split) items on the GPU, full
// splits first and partial last splits from the largest down, so that the
// grid's in-order dispatch ends on its shortest items (decode_items_kernel).
// Each record carries the request's query token, visible range and the
// split's key range, so a workgroup needs no metadata loads of its own.
//
// Per 16-token tile a wave computes S^T = K . Q^T with v_mfma_f32_16x16x32
// (M = 16 tokens, N = the G query heads of the KV head, padded to 16,
// K = head_dim), so K is consumed straight from its natural
// row layout. The softmax runs on the accumulator layout (each lane holds 4
// tokens of one head: max/sum need only two cross-lane steps). P^T is
// already the B operand of O^T += V^T . P^T (v_mfma_f32_16x16x16), which
// keeps alpha rescaling in-lane; V^T comes from a transposed read of the V
// tile through a per-wave LDS slab. P is fed as a bf16 hi/lo pair so the
// P.V product keeps ~16 mantissa bits (the kernel is HBM-bound; the extra
// MFMAs are free).
//
// Each split writes (max, sum, unnormalised acc) partials; a request whose
// context fits one split writes its output directly. The workgroup that
// completes a request merges its partials with the standard log-sum-exp
// rescaling (FlashAttention-2, Dao 2023; flash-decoding, Dao et al. 2023).
// The grid's last workgroups fill the rows that no split writes.
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include <hip/hip_ext.h>

#include "decode_split.h"

namespace mvllm {
namespace {

using namespace dec;

constexpr int kDim = 128;  // head_dim of the general kernel
constexpr int kRow = 144;  // LDS row stride (elements): 288 B keeps both LDS access patterns conflict-free
constexpr int kMaxWaves = 8;

// One 16-token tile of one KV head as MFMA A operands: lane (col, grp)
// holds token `col`, dims 32i + 8grp .. +8 of K and of V.
struct Tile {
  short8_t k[4];
  short8_t v[4];
  bool ok;
};

template <bool NT>
__device__ __forceinline__ short8_t load16(const uint16_t* p) {
  if constexpr (NT) {
    return __builtin_nontemporal_load(reinterpret_cast<const short8_t*>(p));
  } else {
    return *reinterpret_cast<const short8_t*>(p);
  }
}

template <bool NT>
__device__ __forceinline__ void load_tile(const AttnArgs& a, const uint16_t* cache, int64_t r,
                                          int64_t base, int64_t lo, int64_t end, int col,
                                          int64_t head_off, Tile& t) {
  const int64_t tk = base + col;
  bool ok = tk >= lo && tk <= end;
  int64_t off = 0;
  if (ok) {
    const int64_t b = block_of(a, r, tk);
    ok = b >= 0;
    off = b * a.c_s[1] + (tk % a.block_size) * a.c_s[2] + head_off;
  }
  const short8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    t.k[i] = ok ? load16<NT>(cache + off + 32 * i) : zero;
    t.v[i] = ok ? load16<NT>(cache + a.c_s[0] + off + 32 * i) : zero;
  }
  t.ok = ok;
}

template <typename T, bool PREFETCH, bool NT>
__global__ __launch_bounds__(512) void decode_split_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[kMaxWaves][16 * kRow];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int col = lane & 15;
  const int grp = lane >> 4;
  const int waves = blockDim.x >> 6;
  // 1-D grid: workgroup b takes head group b % groups of work-list slot b / groups.
  const int groups = (a.num_kv_heads + waves - 1) / waves;
  const int h = static_cast<int>(blockIdx.x % groups) * waves + wave;
  const int64_t slot = blockIdx.x / groups;
  if (slot >= a.item_capacity) {  // past the work list's capacity
    tidy_rows<T>(a, static_cast<int64_t>(blockIdx.x) - a.item_capacity * groups);
    return;
  }
  const DecodeItem item = a.decode_items[slot];
  if (item.r < 0 || item.r >= a.num_requests) return;
  const int split = item.split;
  const int64_t r = item.r;
  const bool live = h < a.num_kv_heads;  // a spare wave only joins the epilogue's barriers
  const int64_t qs = item.qs;
  const int64_t lo = item.lo;
  const int64_t begin = item.begin;
  const int64_t end = live ? item.end : item.begin - 1;
  // Records index the query, the table and the partials: out-of-range
  // fields (never written by the work-list kernel) end the workgroup.
  if (begin < 0 || begin > item.end || end - begin >= a.split_tokens || end >= a.width * a.block_size ||
      qs < 0 || qs >= a.num_tokens || split < 0 || split >= item.ns || item.base < 0 ||
      static_cast<int64_t>(item.base) + item.ns > a.item_capacity)
    return;

  // Q^T as the B operand: lane (col, grp) holds head col, dims 32i + 8grp .. +8.
  const int G = a.group;
  const int hq = h * G + col;
  short8_t qv[4];
  {
    const uint16_t* qp = static_cast<const uint16_t*>(a.q) + qs * a.q_s0 +
                         static_cast<int64_t>(live && col < G ? hq : 0) * a.q_s1 + 8 * grp;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      qv[i] = (live && col < G) ? *reinterpret_cast<const short8_t*>(qp + 32 * i) : short8_t{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }

  float4_t acc[kDim / 16];
#pragma unroll
  for (int b = 0; b < kDim / 16; ++b) acc[b] = float4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  uint16_t* slab = lds[wave];
  const uint16_t* cache = static_cast<const uint16_t*>(a.cache);
  const int64_t head_off = static_cast<int64_t>(h) * kDim + 8 * grp;

  Tile cur;
  load_tile<NT>(a, cache, r, begin, lo, end, col, head_off, cur);
  for (int64_t base = begin; base <= end; base += 16) {
    Tile nxt;
    if constexpr (PREFETCH) {
      if (base + 16 <= end) load_tile<NT>(a, cache, r, base + 16, lo, end, col, head_off, nxt);
    }
    const uint64_t okmask = __ballot(cur.ok);  // bit j (j < 16): token j of the tile is visible

    float4_t sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) sc = Mfma<T>::k32(cur.k[i], qv[i], sc);

    float s[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      s[e] = ((okmask >> (4 * grp + e)) & 1u) ? sc[e] * a.scale_log2 : -INFINITY;
    float bm = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
    bm = max_xor32_f(max_xor16_f(bm));
    const float mn = fmaxf(m, bm);
    const float alpha = (mn == -INFINITY) ? 1.f : exp2f(m - mn);
    float p[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = (s[e] == -INFINITY) ? 0.f : exp2f(s[e] - mn);
    l = l * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
    if (__ballot(alpha != 1.f)) {
#pragma unroll
      for (int b = 0; b < kDim / 16; ++b) acc[b] *= alpha;
    }
    m = mn;

    // P^T as the B operand (tokens 4grp .. +4 of head col), as a hi/lo pair.
    uint32_t ph[4], pl[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) split_hi_lo<T>(p[e], ph[e], pl[e]);
    const short4_t pb_hi = __builtin_bit_cast(short4_t, uint2{ph[0] | (ph[1] << 16), ph[2] | (ph[3] << 16)});
    const short4_t pb_lo = __builtin_bit_cast(short4_t, uint2{pl[0] | (pl[1] << 16), pl[2] | (pl[3] << 16)});

    // V tile -> LDS (row = token, natural layout), then read V^T.
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<short8_t*>(slab + col * kRow + 32 * i + 8 * grp) = cur.v[i];
    wave_lds_sync();
#pragma unroll
    for (int b = 0; b < kDim / 16; ++b) {
      // A operand: lane (col, grp) receives V[token 4grp + e][dim 16b + col].
      const uint32_t at = lds_address(slab + (4 * grp + (col >> 2)) * kRow + 16 * b + 4 * (col & 3));
      const short4_t av = __builtin_bit_cast(
          short4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_tr_short4*>(static_cast<uintptr_t>(at))));
      acc[b] = Mfma<T>::k16(av, pb_hi, acc[b]);
      acc[b] = Mfma<T>::k16(av, pb_lo, acc[b]);
    }
    if constexpr (PREFETCH) {
      cur = nxt;
    } else {
      if (base + 16 <= end) load_tile<NT>(a, cache, r, base + 16, lo, end, col, head_off, cur);
    }
  }

  const float lt = sum_xor32_f(sum_xor16_f(l));
  // A launch of its own merges: with the merge here the kernel needs 236
  // registers instead of 138 and runs two waves per SIMD instead of three (23
  // contexts of up to 28,670 in blocks of 8: 491 us before, 601 with it).
  finish_split<T, kDim, false>(a, item, h, live, static_cast<int>(blockIdx.x % groups), groups, m, lt, acc, nullptr);
}

// The pipelined kernel (decode_split_lds_body) for block sizes that are
// multiples of 16: K and V tiles go straight from HBM to LDS.
template <typename T, int D, int STAGES>
__global__ __launch_bounds__(256, 2) void decode_split_lds_kernel(AttnArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  decode_split_lds_body<T, D, STAGES>(a, smem, blockIdx.x, blockDim.x >> 6);
}


// The merge as a launch of its own: a workgroup of four waves takes
// kMergeHeads query heads of one request, two per wave.
constexpr int kMergeHeads = 8;

template <typename T, int D>
__global__ __launch_bounds__(256) void decode_merge_kernel(AttnArgs a, int32_t head_blocks) {
  const int64_t r = blockIdx.x / head_blocks;
  const int2 req = a.decode_req[r];  // (query token, splits)
  const int64_t base = a.done[r];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int head0 = static_cast<int>(blockIdx.x % head_blocks) * kMergeHeads + 2 * wave;
  if (req.y <= 1 || req.x < 0 || req.x >= a.num_tokens || base < 0 || base + req.y > a.item_capacity ||
      head0 >= a.num_q_heads)
    return;
  merge_request<T, D>(a, base, req.x, head0, a.num_q_heads - head0 < 2 ? 1 : 2, req.y);
}

__global__ __launch_bounds__(kDecodeListThreads) void decode_items_kernel(AttnArgs a) { build_decode_list(a); }

struct DecodeTuning {
  bool lds_pipeline;  // the global->LDS pipelined kernel (block_size % 16 == 0)
  int waves;          // waves (KV heads) per workgroup
  int stages;         // tiles in flight per wave (pipelined kernel)
  bool prefetch;      // register prefetch (general kernel)
  bool nontemporal;   // non-temporal loads (general kernel)
};

DecodeTuning decode_tuning(const AttnArgs& a) {
  DecodeTuning t;
  t.lds_pipeline = !decode_general(a);
  t.waves = 4;
  t.stages = a.head_dim == 64 ? kStages<64> : a.head_dim == 96 ? kStages<96> : kStages<128>;
  t.prefetch = false;
  t.nontemporal = false;
  if (const char* env = std::getenv("MVLLM_DECODE_WAVES")) {
    const int v = std::atoi(env);
    if (v >= 1 && v <= kMaxWaves) t.waves = v;
  }
  if (const char* env = std::getenv("MVLLM_DECODE_STAGES")) {
    const int v = std::atoi(env);
    if (v >= 2 && v <= 4 && a.head_dim == kDim) t.stages = v;
  }
  if (const char* env = std::getenv("MVLLM_DECODE_PREFETCH")) t.prefetch = std::atoi(env) != 0;
  if (const char* env = std::getenv("MVLLM_DECODE_NT")) t.nontemporal = std::atoi(env) != 0;
  if (t.lds_pipeline && t.waves > 4) t.waves = 4;
  if (t.waves > a.num_kv_heads) t.waves = a.num_kv_heads;
  return t;
}

template <typename T, int D, int STAGES>
int launch_lds_kernel(const AttnArgs& a, dim3 grid, int waves, hipStream_t s, hipEvent_t start,
                      hipEvent_t stop) {
  const size_t lds = static_cast<size_t>(waves) * STAGES * 2 * kTileBytesOf<D>;
  if (lds > 64 * 1024) {
    static bool raised = false;  // per instantiation; the attribute is process-wide
    if (!raised) {
      MVLLM_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(decode_split_lds_kernel<T, D, STAGES>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        static_cast<int>(lds)));
      raised = true;
    }
  }
  hipExtLaunchKernelGGL((decode_split_lds_kernel<T, D, STAGES>), grid, dim3(64 * waves), lds, s, start, stop,
                        0, a);
  MVLLM_LAUNCH_CHECK("decode_split_lds_kernel");
  return MVLLM_OK;
}

template <typename T, int D>
int launch_merge_t(const AttnArgs& a, hipStream_t s) {
  const int32_t head_blocks = (a.num_q_heads + kMergeHeads - 1) / kMergeHeads;
  const int64_t blocks = a.num_requests * head_blocks;
  if (blocks > INT32_MAX) return fail(MVLLM_ERR_INVALID, "merge grid too large (%lld workgroups)", (long long)blocks);
  hipLaunchKernelGGL((decode_merge_kernel<T, D>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, a, head_blocks);
  MVLLM_LAUNCH_CHECK("decode_merge_kernel");
  return MVLLM_OK;
}

template <typename T, int D>
int launch_decode_t(const AttnArgs& a, hipStream_t s, hipEvent_t start, hipEvent_t stop) {
  const DecodeTuning tune = decode_tuning(a);
  const int waves = tune.waves;
  const int groups = (a.num_kv_heads + waves - 1) / waves;

  if (a.num_requests > 0) {
    const int64_t blocks = a.item_capacity * groups + tidy_blocks(a);
    if (blocks > INT32_MAX) return fail(MVLLM_ERR_INVALID, "decode grid too large (%lld workgroups)", (long long)blocks);
    if (!a.lists_ready) {
      if (int rc = launch_decode_lists(a, s)) return rc;
    } else if (a.width * a.block_size > INT32_MAX || a.num_tokens > INT32_MAX) {
      return fail(MVLLM_ERR_UNSUPPORTED, "decode positions beyond 2^31 are not supported");
    }
    const dim3 grid(static_cast<unsigned>(blocks));
    const dim3 block(64 * waves);
    if constexpr (D != kDim) {
      if (!tune.lds_pipeline)
        return fail(MVLLM_ERR_UNSUPPORTED, "head_dim %d needs block sizes that are multiples of 16", D);
      if (int rc = launch_lds_kernel<T, D, kStages<D>>(a, grid, waves, s, start, stop)) return rc;
    } else if (tune.lds_pipeline) {
      int rc = MVLLM_OK;
      if (tune.stages == 2) rc = launch_lds_kernel<T, D, 2>(a, grid, waves, s, start, stop);
      else if (tune.stages == 3) rc = launch_lds_kernel<T, D, 3>(a, grid, waves, s, start, stop);
      else rc = launch_lds_kernel<T, D, 4>(a, grid, waves, s, start, stop);
      if (rc) return rc;
    } else {
      if (tune.prefetch && tune.nontemporal)
        hipExtLaunchKernelGGL(decode_split_kernel<T, true, true>, grid, block, 0, s, start, stop, 0, a);
      else if (tune.prefetch)
        hipExtLaunchKernelGGL(decode_split_kernel<T, true, false>, grid, block, 0, s, start, stop, 0, a);
      else if (tune.nontemporal)
        hipExtLaunchKernelGGL(decode_split_kernel<T, false, true>, grid, block, 0, s, start, stop, 0, a);
      else
        hipExtLaunchKernelGGL(decode_split_kernel<T, false, false>, grid, block, 0, s, start, stop, 0, a);
      MVLLM_LAUNCH_CHECK("decode_split_kernel");
    }
  }
  return MVLLM_OK;
}

// Calls f(T{}, integral_constant D) for the decode kernels' types and head
// dims; `unsupported` for any other.
template <typename F>
int for_decode_types(const AttnArgs& a, int32_t dtype, F&& f) {
  auto dims = [&](auto t) {
    if (a.head_dim == 128) return f(t, std::integral_constant<int, 128>{});
    if (a.head_dim == 96) return f(t, std::integral_constant<int, 96>{});
    if (a.head_dim == 64) return f(t, std::integral_constant<int, 64>{});
    return fail(MVLLM_ERR_UNSUPPORTED, "decode kernel needs head_dim 64, 96 or 128");
  };
  if (dtype == MVLLM_DTYPE_BF16) return dims(bf16_t{});
  if (dtype == MVLLM_DTYPE_F16) return dims(f16_t{});
  return fail(MVLLM_ERR_UNSUPPORTED, "decode kernel needs bf16 or fp16");
}

}  // namespace

int launch_decode_lists(const AttnArgs& a, hipStream_t s) {
  if (a.num_requests <= 0) return MVLLM_OK;
  if (!a.decode_items || !a.decode_req) return fail(MVLLM_ERR_INVALID, "decode work list is missing");
  // Work-list records carry positions and token indices as int32.
  if (a.width * a.block_size > INT32_MAX || a.num_tokens > INT32_MAX)
    return fail(MVLLM_ERR_UNSUPPORTED, "decode positions beyond 2^31 are not supported");
  hipLaunchKernelGGL(decode_items_kernel, dim3(1), dim3(kDecodeListThreads), 0, s, a);
  MVLLM_LAUNCH_CHECK("decode_items_kernel");
  return MVLLM_OK;
}

int launch_decode(const AttnArgs& a, int32_t dtype, hipStream_t s, hipEvent_t start,
                  hipEvent_t stop) {
  if (int rc = for_decode_types(a, dtype, [&](auto t, auto d) {
        return launch_decode_t<decltype(t), decltype(d)::value>(a, s, start, stop);
      }))
    return rc;
  return launch_merge(a, dtype, s);
}

int launch_merge(const AttnArgs& a, int32_t dtype, hipStream_t s) {
  if (!a.merge_apart || a.num_requests <= 0) return MVLLM_OK;
  return for_decode_types(a, dtype, [&](auto t, auto d) { return launch_merge_t<decltype(t), decltype(d)::value>(a, s); });
}

bool decode_supported(int64_t head_dim, int64_t block_size, int64_t split_tokens) {
  return head_dim == 128 || ((head_dim == 64 || head_dim == 96) && block_size % 16 == 0 && split_tokens <= kMaxSplit);
}

bool decode_general(const AttnArgs& a) {
  if (a.block_size % 16 != 0 || a.split_tokens > kMaxSplit || !rows_within_32_bits(a.c_s[2])) return true;
  // The general kernel exists at head_dim 128 only.
  const char* env = std::getenv("MVLLM_DECODE_KERNEL");
  return env && std::strcmp(env, "general") == 0 && a.head_dim == kDim;
}

bool decode_step_eligible(const AttnArgs& a) {
  if (!decode_supported(a.head_dim, a.block_size, a.split_tokens) || a.num_requests <= 0) return false;
  // The default shape only (fewer KV heads than waves: the spare waves of
  // the step's workgroups end at once, as the pipelined kernel's do).
  const DecodeTuning tune = decode_tuning(a);
  const int waves = a.num_kv_heads < kStepDecodeWaves ? a.num_kv_heads : kStepDecodeWaves;
  return tune.lds_pipeline && tune.waves == waves && (a.head_dim != 128 || tune.stages == kStages<128>);
}

int64_t decode_step_blocks(const AttnArgs& a) {
  return a.item_capacity * ((a.num_kv_heads + kStepDecodeWaves - 1) / kStepDecodeWaves) + tidy_blocks(a);
}

}  // namespace mvllm
