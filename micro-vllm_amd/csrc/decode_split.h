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
// bits; the V^T operand comes from transposing LDS reads (ds_read_b64_tr_b16).
#pragma once

#include <cmath>

#include "worklists.h"

namespace mvllm {
namespace {
namespace dec {

template <typename T>
__device__ __forceinline__ void split_hi_lo(float p, uint32_t& hi, uint32_t& lo) {
  hi = Elem<T>::to_bits(p);
  lo = Elem<T>::to_bits(p - Elem<T>::from_bits(hi));
}

// Epilogue shared by the decode kernels. acc[b][e] is
// O[head hq][dim 16b + 4grp + e] (unnormalised), m / lt the running
// max (exp2 domain) and the complete softmax denominator of this split. A
// request with one split gets its output directly; otherwise the partial goes
// to the workspace for the combine kernel.
template <typename T, int D>
__device__ __forceinline__ void write_decode_result(const AttnArgs& a, int64_t r, int64_t qs, int hq,
                                                    int split, int64_t ns, float m, float lt,
                                                    const float4_t (&acc)[D / 16], int grp) {
  if (ns == 1) {
    const float inv = 1.f / lt;
    uint16_t* op = static_cast<uint16_t*>(a.out) + qs * a.o_s0 + static_cast<int64_t>(hq) * a.o_s1;
#pragma unroll
    for (int b = 0; b < D / 16; ++b) {
      const uint32_t w0 = Elem<T>::to_bits(acc[b][0] * inv) | (Elem<T>::to_bits(acc[b][1] * inv) << 16);
      const uint32_t w1 = Elem<T>::to_bits(acc[b][2] * inv) | (Elem<T>::to_bits(acc[b][3] * inv) << 16);
      *reinterpret_cast<uint2*>(op + 16 * b + 4 * grp) = uint2{w0, w1};
    }
    return;
  }
  const int64_t item = (r * a.max_splits + split) * a.num_q_heads + hq;
  float* wp = a.ws_acc + item * D;
#pragma unroll
  for (int b = 0; b < D / 16; ++b) *reinterpret_cast<float4_t*>(wp + 16 * b + 4 * grp) = acc[b];
  if (grp == 0) a.ws_ml[item] = float2{m, lt};
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
// block ids are fetched once, up front). The loads carry the non-temporal
// hint: every K/V byte is read exactly once, and keeping the stream from
// displacing other cached lines raised the measured bandwidth from 5.5 to
// 6.0 TB/s on the Qwen3 decode batch.

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

template <typename T, int D, int STAGES>
__device__ __forceinline__ void decode_split_lds_body(const AttnArgs& a, uint8_t* smem, uint32_t wg, int waves) {
  constexpr int kTileBytes = kTileBytesOf<D>;
  constexpr int kLoads = D / 32;  // 1 KiB loads per K (or V) tile
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int col = lane & 15;
  const int grp = lane >> 4;
  // 1-D grid: workgroup b takes head group b % groups of work-list slot b / groups.
  const int groups = (a.num_kv_heads + waves - 1) / waves;
  const int h = static_cast<int>(wg % groups) * waves + wave;
  // The work-list record carries the request's query token, visible range
  // and this split's key range, so the first tile loads wait on two
  // dependent loads (the record, then the block ids) rather than four.
  const DecodeItem item = a.decode_items[wg / groups];
  if (item.r < 0 || item.r >= a.num_requests) return;
  if (h >= a.num_kv_heads) return;
  const int split = item.split;
  const int64_t r = item.r;
  const int64_t qs = item.qs;
  const int64_t lo = item.lo;
  const int64_t begin = item.begin;
  const int64_t end = item.end;
  // Records index the query, the table and the partials: out-of-range
  // fields (never written by the work-list kernel) end the workgroup.
  if (begin < 0 || begin > end || end - begin >= a.split_tokens || end >= a.width * a.block_size ||
      qs < 0 || qs >= a.num_tokens || split < 0 || split >= a.max_splits)
    return;
  const int ntiles = static_cast<int>((end - begin) / 16 + 1);  // <= 128 (split <= 2048)

  // Block id and in-block row of tiles `lane` and `lane + 64` of this split,
  // fetched once (block ids are < 2^31; a 16-aligned tile never straddles a
  // block).
  int32_t my_block[2] = {-1, -1}, my_row[2] = {0, 0};
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    if (lane + 64 * x < ntiles) {
      const int64_t p = begin + 16 * (lane + 64 * x);
      my_block[x] = static_cast<int32_t>(block_of(a, r, p));
      my_row[x] = static_cast<int32_t>(p % a.block_size);
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
                         static_cast<int64_t>(col < G ? hq : 0) * a.q_s1 + 8 * grp;
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      qv[i] = (col < G) ? *reinterpret_cast<const short8_t*>(qp + 32 * i) : short8_t{0, 0, 0, 0, 0, 0, 0, 0};
  }

  uint8_t* wave_lds = smem + static_cast<size_t>(wave) * STAGES * 2 * kTileBytes;
  const uint32_t wave_lds_addr = lds_address(wave_lds);
  const uint16_t* cache = static_cast<const uint16_t*>(a.cache);
  const int64_t head_elems = static_cast<int64_t>(h) * D;

  // Load-side mapping: instruction i, this lane -> 16-byte chunk 64i + lane of
  // the tile's LDS slot (element offset of its data from the tile's first row).
  int64_t lane_off[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int t = (64 * i + lane) / (D / 8);
    const int p = (64 * i + lane) % (D / 8);
    lane_off[i] = t * a.c_s[2] + 8 * tile_logical<D>(t, p);
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
    const uint32_t kdst = wave_lds_addr + stage * 2 * kTileBytes;
    const uint32_t vdst = kdst + kTileBytes;
    // An invalid block id masks the whole tile: read a valid dummy line instead.
    const uint16_t* tile_k = blk >= 0 ? cache + static_cast<int64_t>(blk) * a.c_s[1] +
                                            static_cast<int64_t>(row) * a.c_s[2] + head_elems
                                      : cache;
    const int64_t plane = blk >= 0 ? a.c_s[0] : 0;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const uint16_t* src = blk >= 0 ? tile_k + lane_off[i] : cache;
      lds_dma_load16_stream(src, kdst + i * 1024);
      lds_dma_load16_stream(src + plane, vdst + i * 1024);
    }
  };

  float4_t acc[D / 16];
#pragma unroll
  for (int b = 0; b < D / 16; ++b) acc[b] = float4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  // The block ids and Q must be in registers before the first tile address.
  __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < ntiles) issue(s, s);

  for (int k = 0; k < ntiles; ++k) {
    const int stage = k % STAGES;
    const int ahead = k + STAGES - 1;
    if (ahead < ntiles) {
      // The stage being refilled, (k - 1) % STAGES, was read in the previous
      // iteration. Its LDS reads have retired only because that iteration
      // ended with an lgkmcnt(0) wait; that wait is what makes the refill safe.
      issue(ahead, ahead % STAGES);
    }
    const int later = (ntiles - 1 - k) < (STAGES - 1) ? (ntiles - 1 - k) : (STAGES - 1);
    wait_tiles<2 * kLoads>(later);
    __builtin_amdgcn_wave_barrier();
    compiler_fence();

    const int64_t tb = begin + 16 * static_cast<int64_t>(k);
    const int64_t blk = tile_block(k);
    // Token j of the tile is visible iff its position is in [lo, end] and the block is valid.
    uint32_t okmask = 0;
    if (blk >= 0) {
      const int64_t first_ok = lo > tb ? lo - tb : 0;
      const int64_t last_ok = end - tb < 15 ? end - tb : 15;
      okmask = (last_ok >= first_ok) ? ((0xFFFFu >> (15 - last_ok)) & (0xFFFFu << first_ok)) : 0u;
    }
    const uint8_t* kt = wave_lds + stage * 2 * kTileBytes;
    const uint32_t vt = wave_lds_addr + stage * 2 * kTileBytes + kTileBytes;

    float4_t sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const short8_t kk = *reinterpret_cast<const short8_t*>(kt + koff[i]);
      sc = Mfma<T>::k32(kk, qv[i], sc);
    }
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
      for (int b = 0; b < D / 16; ++b) acc[b] *= alpha;
    }
    m = mn;

    uint32_t ph[4], pl[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) split_hi_lo<T>(p[e], ph[e], pl[e]);
    const short4_t pb_hi = __builtin_bit_cast(short4_t, uint2{ph[0] | (ph[1] << 16), ph[2] | (ph[3] << 16)});
    const short4_t pb_lo = __builtin_bit_cast(short4_t, uint2{pl[0] | (pl[1] << 16), pl[2] | (pl[3] << 16)});
    // Rows of masked tokens may hold stale or non-finite data: zero them in V.
    const uint32_t mlo = ((okmask >> (4 * grp)) & 1u ? 0xFFFFu : 0u) | ((okmask >> (4 * grp + 1)) & 1u ? 0xFFFF0000u : 0u);
    const uint32_t mhi = ((okmask >> (4 * grp + 2)) & 1u ? 0xFFFFu : 0u) | ((okmask >> (4 * grp + 3)) & 1u ? 0xFFFF0000u : 0u);
#pragma unroll
    for (int b = 0; b < D / 16; ++b) {
      // A operand: lane (col, grp) receives V[token 4grp + e][dim 16b + col].
      const uint2 rv = __builtin_bit_cast(
          uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_tr_short4*>(static_cast<uintptr_t>(vt + voff[b]))));
      const short4_t av = __builtin_bit_cast(short4_t, uint2{rv.x & mlo, rv.y & mhi});
      acc[b] = Mfma<T>::k16(av, pb_hi, acc[b]);
      acc[b] = Mfma<T>::k16(av, pb_lo, acc[b]);
    }
    // All LDS reads of this stage must retire before a later issue refills it.
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    compiler_fence();
  }

  const float lt = sum_xor32_f(sum_xor16_f(l));
  if (col >= G) return;
  write_decode_result<T, D>(a, r, qs, hq, split, item.ns, m, lt, acc, grp);
}

}  // namespace dec
}  // namespace
}  // namespace mvllm
