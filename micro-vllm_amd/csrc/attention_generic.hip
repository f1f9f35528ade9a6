// The attention kernels outside the 16-bit matrix-core path: fp32 attention on
// the fp32 matrix cores (attention_f32_kernel, below), and any-shape ragged
// paged attention, one workgroup of W waves per (token, query head).
//
// The any-shape kernel carries the shapes the specialised kernels do not
// (other head_dims, query-head groups above 16, non-contiguous rows): each wave walks every W-th block of 64 keys, each lane scoring
// one key, then accumulates P.V with lanes spread over head_dim (one
// instantiation per bound of 64, 128, 256 and 512 elements, so the loops
// over a lane's elements and over a block's keys unroll without guards on
// elements past head_dim's bound). Online softmax in fp32 (exp2 domain) in
// the manner of FlashAttention-2 (Dao, 2023); the waves' partial states are
// merged through LDS at the end, so a long visible range costs 1/W of the
// dependent memory round trips of one wave walking it alone. W is 4 when
// the block table reaches at most 1,024 keys (more waves would find no
// block to walk) and 16 beyond (8 for head_dim above 128, whose
// accumulators do not fit the register share of 16 waves).
#include <climits>
#include <cmath>

#include "attention.h"

namespace mvllm {
namespace {

constexpr int kMaxDimPerLane = 8;  // head_dim <= 512

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
  return v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

// The 16 bytes at p (16-byte aligned) as 16 / sizeof(T) floats.
template <typename T>
__device__ __forceinline__ void load16(const T* p, float (&f)[16 / sizeof(T)]) {
  const uint4 w = *reinterpret_cast<const uint4*>(p);
  const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = __uint_as_float(ws[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = Elem<T>::from_bits(ws[i] & 0xFFFFu);
      f[2 * i + 1] = Elem<T>::from_bits(ws[i] >> 16);
    }
  }
}

// Largest i in [0, R] with qsl[i] <= t (qsl is non-decreasing).
__device__ __forceinline__ int64_t request_of(const AttnArgs& a, int64_t t) {
  int64_t lo = 0, hi = a.num_requests;
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) >> 1;
    if (a.qsl[mid] <= t) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// DPL: head_dim elements per lane in the P.V accumulation (head_dim <= 64 * DPL);
// WAVES: waves per workgroup, each walking every WAVES-th block of 64 keys.
template <typename T, int DPL, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void attention_generic_kernel(AttnArgs a) {
  const int64_t t = blockIdx.x;
  const int hq = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int D = a.head_dim;
  T* out = static_cast<T*>(a.out) + t * a.o_s0 + static_cast<int64_t>(hq) * a.o_s1;

  const int64_t r = request_of(a, t);
  const bool covered = r < a.num_requests && a.qsl[r] <= t && t < a.qsl[r + 1];
  if (!covered) {
    if (a.mode == 0)
      for (int d = threadIdx.x; d < D; d += 64 * WAVES) Elem<T>::store(out + d * a.o_s2, 0.f);
    return;
  }
  const int64_t qs = a.qsl[r];
  if (a.mode == 1 && a.qsl[r + 1] - qs == 1) return;

  __shared__ float qsh[64 * DPL];
  const T* q = static_cast<const T*>(a.q) + t * a.q_s0 + static_cast<int64_t>(hq) * a.q_s1;
  for (int d = threadIdx.x; d < D; d += 64 * WAVES) qsh[d] = Elem<T>::load(q + d * a.q_s2) * a.scale_log2;
  __syncthreads();

  int64_t lo, hi;
  visible_range(a, r, qs, t, lo, hi);
  const int kvh = hq / a.group;
  const T* cache = static_cast<const T*>(a.cache);
  float acc[DPL];
#pragma unroll
  for (int j = 0; j < DPL; ++j) acc[j] = 0.f;
  float m = -INFINITY, l = 0.f;
  // Key rows contiguous and 16-byte aligned: each lane reads its row in
  // 16-byte pieces (a quarter or an eighth of the load instructions, each
  // of which touches one cache line per lane).
  constexpr int kVec = 16 / static_cast<int>(sizeof(T));
  const bool vec_rows = a.c_s[4] == 1 && D % kVec == 0 && a.c_s[1] % kVec == 0 && a.c_s[2] % kVec == 0 &&
                        a.c_s[3] % kVec == 0 && (reinterpret_cast<uintptr_t>(a.cache) & 15u) == 0;

  for (int64_t base = lo + 64 * wave; base <= hi; base += 64 * WAVES) {
    const int64_t p = base + lane;
    int64_t row = -1;  // element offset of this lane's key row
    if (p <= hi) {
      const int64_t b = block_of(a, r, p);
      if (b >= 0)
        row = b * a.c_s[1] + (p % a.block_size) * a.c_s[2] + static_cast<int64_t>(kvh) * a.c_s[3];
    }
    // Four independent partial sums, so a lane keeps several loads of its
    // key row in flight instead of one chain of dependent ones.
    float s = -INFINITY;
    if (row >= 0) {
      const T* kp = cache + row;
      const int64_t ks = a.c_s[4];
      float d0 = 0.f, d1 = 0.f, d2 = 0.f, d3 = 0.f;
      int d = 0;
      if (vec_rows) {
#pragma unroll 16
        for (; d < D; d += kVec) {
          float f[kVec];
          load16(kp + d, f);
#pragma unroll
          for (int e = 0; e < kVec; e += 4) {
            d0 = __builtin_fmaf(qsh[d + e], f[e], d0);
            d1 = __builtin_fmaf(qsh[d + e + 1], f[e + 1], d1);
            d2 = __builtin_fmaf(qsh[d + e + 2], f[e + 2], d2);
            d3 = __builtin_fmaf(qsh[d + e + 3], f[e + 3], d3);
          }
        }
      } else {
#pragma unroll 8
        for (; d + 4 <= D; d += 4) {
          d0 = __builtin_fmaf(qsh[d], Elem<T>::load(kp + d * ks), d0);
          d1 = __builtin_fmaf(qsh[d + 1], Elem<T>::load(kp + (d + 1) * ks), d1);
          d2 = __builtin_fmaf(qsh[d + 2], Elem<T>::load(kp + (d + 2) * ks), d2);
          d3 = __builtin_fmaf(qsh[d + 3], Elem<T>::load(kp + (d + 3) * ks), d3);
        }
        for (; d < D; ++d) d0 = __builtin_fmaf(qsh[d], Elem<T>::load(kp + d * ks), d0);
      }
      s = (d0 + d1) + (d2 + d3);
    }
    const float mn = fmaxf(m, wave_max(s));
    const float alpha = (mn == -INFINITY) ? 1.f : exp2f(m - mn);
    const float pr = (s == -INFINITY) ? 0.f : exp2f(s - mn);
    l = l * alpha + wave_sum(pr);
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] *= alpha;
    // P.V without a branch per key, so the loads of several keys overlap:
    // a key with no row reads row 0 of the V plane and adds nothing (a
    // select, not a product with 0, so a non-finite stale value stays out).
    const int count = static_cast<int>(hi - base + 1 < 64 ? hi - base + 1 : 64);
#pragma unroll 32
    for (int k = 0; k < count; ++k) {
      const int64_t vrow = __shfl(row, k, 64);
      const float pk = __shfl(pr, k, 64);
      const bool has = vrow >= 0;
      const T* vp = cache + a.c_s[0] + (has ? vrow : 0);
#pragma unroll
      for (int j = 0; j < DPL; ++j) {
        const int d = lane + 64 * j;
        if (d < D) {
          const float pv = pk * Elem<T>::load(vp + d * a.c_s[4]);
          acc[j] += has ? pv : 0.f;
        }
      }
    }
    m = mn;
  }
  // Merge the waves' (offset, sum, accumulator) states; a wave that saw no
  // key holds (-inf, 0, 0) and weighs nothing.
  __shared__ float msh[WAVES], lsh[WAVES];
  __shared__ float accsh[WAVES][64 * DPL];
  if (lane == 0) {
    msh[wave] = m;
    lsh[wave] = l;
  }
#pragma unroll
  for (int j = 0; j < DPL; ++j) {
    const int d = lane + 64 * j;
    if (d < D) accsh[wave][d] = acc[j];
  }
  __syncthreads();
  if (wave != 0) return;
  float mx = -INFINITY;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) mx = fmaxf(mx, msh[w]);
  float weight[WAVES];
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    weight[w] = msh[w] == -INFINITY ? 0.f : exp2f(msh[w] - mx);
    total += weight[w] * lsh[w];
  }
  const float inv = 1.f / total;  // an empty visible range gives 0/0 = NaN, as the reference's softmax does
#pragma unroll
  for (int j = 0; j < DPL; ++j) {
    const int d = lane + 64 * j;
    if (d < D) {
      float o = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) o += weight[w] * accsh[w][d];
      Elem<T>::store(out + d * a.o_s2, o * inv);
    }
  }
}

// fp32 attention on the fp32 matrix cores (head_dim 64 or 128, up to 16 query
// heads per KV head, contiguous 16-byte aligned rows).
//
// A workgroup of eight waves takes one KV head and a block of T = 16 / G tokens
// of one request: the 16 columns of v_mfma_f32_16x16x4_f32 are its (query head
// of the group, token) pairs, so the group's heads and a chunk's neighbouring
// tokens read each key once. Each wave walks every eighth tile of 16 keys, K
// and V loaded straight into the operand registers in 16-byte pieces, the next
// tile's while one is computed: S^T = K . Q^T with k index `grp` of step
// (i, s) standing for dim 16 i + 4 grp + s on both sides, so a lane's four
// steps come from one piece; the accumulator holds tokens 4 grp + e, which is
// the B operand of O^T += V^T . P^T with token 4 grp + s at step s, whose A
// operand is a lane's piece of row 4 grp + s (column m of block (j, c) is dim
// 64 j + 4 m + c). Products, probabilities and sums are fp32 throughout, as in
// the any-shape kernel. The waves' states merge through LDS.
//
// These batches are small and the bound is latency: the any-shape kernel chains
// a binary search, a score per lane over its own row and 64 shuffled V rows per
// block (25.4 us for three decodes and a 17-token prompt of up to 255 keys; 13-14
// here).
constexpr int kTileWaves = 8;
constexpr int kTidyRows = 64;  // tokens per workgroup that clears rows outside every request

// The request whose query blocks contain slot j: block b of request r (first
// query qs) is slot qs / T + r + b. A 64-ary search, one round of loads per
// level; the last level's loads also give the request's query range [qs, qe).
__device__ __forceinline__ int64_t slot_owner(const AttnArgs& a, int64_t slot, int32_t T, int64_t& qs, int64_t& qe) {
  const int lane = threadIdx.x & 63;
  int64_t lo = 0, n = a.num_requests;
  while (true) {
    const int64_t step = (n + 63) / 64;
    const int64_t r = lo + lane * step;
    const bool in = r < lo + n;
    const int64_t mine = a.qsl[in ? r : lo], next = a.qsl[(in ? r : lo) + 1];
    const int count = __popcll(__ballot(in && mine / T + r <= slot));
    if (count == 0) return -1;
    const int64_t at = lo + (count - 1) * step;
    n = lo + n - at < step ? lo + n - at : step;
    lo = at;
    if (n > 1) continue;
    qs = __shfl(mine, count - 1, 64);
    qe = __shfl(next, count - 1, 64);
    return lo;
  }
}

template <int D>
__global__ __launch_bounds__(64 * kTileWaves) void attention_f32_kernel(AttnArgs a, int32_t T, int64_t slots) {
  constexpr int J = D / 64;
  constexpr int kColStride = D + 4;
  __shared__ __attribute__((aligned(16))) float buf[kTileWaves / 2][16 * kColStride];
  __shared__ float msh[kTileWaves][16], lsh[kTileWaves][16];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15;
  const int grp = lane >> 4;
  const int h = blockIdx.y;
  const int G = a.group;
  const int64_t slot = blockIdx.x;
  if (slot >= slots) {
    const int64_t first = a.qsl[0], last = a.qsl[a.num_requests];
    const int64_t t0 = (slot - slots) * kTidyRows;
    for (int64_t t = t0; t < t0 + kTidyRows && t < a.num_tokens; ++t) {
      if (t >= first && t < last) continue;
      for (int i = tid; i < G * D; i += 64 * kTileWaves)
        static_cast<float*>(a.out)[t * a.o_s0 + (static_cast<int64_t>(h) * G + i / D) * a.o_s1 + (i % D) * a.o_s2] = 0.f;
    }
    return;
  }
  int64_t qs = 0, qe = 0;
  const int64_t r = slot_owner(a, slot, T, qs, qe);
  if (r < 0) return;
  if (qe > a.num_tokens) qe = a.num_tokens;
  const int64_t t0 = qs + (slot - (qs / T + r)) * T;
  if (qs < 0 || t0 >= qe) return;

  // This lane's column: (query head g of the group, token tk).
  const int g = col / T;
  const int64_t tk = t0 + col % T;
  const bool column = g < G && tk < qe;
  const int64_t hq = static_cast<int64_t>(h) * G + (column ? g : 0);
  int32_t lo = 1, hi = 0;
  {
    int64_t lo64, hi64;
    visible_range(a, r, qs, column ? tk : t0, lo64, hi64);
    if (column && hi64 >= lo64) {
      lo = static_cast<int32_t>(lo64);
      hi = static_cast<int32_t>(hi64);
    }
  }
  float4_t qf[D / 16];
  {
    const float* qp = static_cast<const float*>(a.q) + (column ? tk : t0) * a.q_s0 + hq * a.q_s1 + 4 * grp;
#pragma unroll
    for (int i = 0; i < D / 16; ++i) qf[i] = *reinterpret_cast<const float4_t*>(qp + 16 * i);
  }
  const bool any = hi >= lo;
  const int32_t first_key = wave_reduce_i(any ? lo : INT32_MAX, [](int32_t x, int32_t y) { return x < y ? x : y; });
  const int32_t last_key = wave_reduce_i(any ? hi : -1, [](int32_t x, int32_t y) { return x > y ? x : y; });
  const int32_t base = first_key & ~15;
  const int32_t ntiles = last_key >= 0 ? (last_key - base) / 16 + 1 : 0;

  const float* const cache = static_cast<const float*>(a.cache) + static_cast<int64_t>(h) * a.c_s[3];
  const uint32_t bs = static_cast<uint32_t>(a.block_size);
  // A tile in registers: this lane's row offset (-1: no such key), K of row
  // `col` and V of rows 4 grp + s. Rows that do not exist read block 0.
  struct Tile {
    bool mapped;
    float4_t k[D / 16], v[4][J];
  };
  auto load = [&](int32_t tile, Tile& t) {
    const uint32_t pos = static_cast<uint32_t>(base + 16 * tile + col);
    int64_t off = -1;
    if (static_cast<int32_t>(pos) >= first_key && static_cast<int32_t>(pos) <= last_key) {
      const int64_t b = a.table[r * a.t_s0 + static_cast<int64_t>(pos / bs) * a.t_s1];
      if (b >= 0 && b < a.num_blocks) off = b * a.c_s[1] + static_cast<int64_t>(pos % bs) * a.c_s[2];
    }
    t.mapped = off >= 0;
    const float* kp = cache + (off >= 0 ? off : 0) + 4 * grp;
#pragma unroll
    for (int i = 0; i < D / 16; ++i) t.k[i] = *reinterpret_cast<const float4_t*>(kp + 16 * i);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int64_t voff = __shfl(off, 4 * grp + s, 64);
      const float* vp = cache + a.c_s[0] + (voff >= 0 ? voff : 0) + 4 * col;
#pragma unroll
      for (int j = 0; j < J; ++j) t.v[s][j] = *reinterpret_cast<const float4_t*>(vp + 64 * j);
    }
  };

  float4_t acc[J][4];
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[j][c] = float4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  Tile cur;
  if (wave < ntiles) load(wave, cur);
  for (int32_t tile = wave; tile < ntiles; tile += kTileWaves) {
    Tile nxt;
    if (tile + kTileWaves < ntiles) load(tile + kTileWaves, nxt);
    const uint32_t mapped = static_cast<uint32_t>(__ballot(cur.mapped)) & 0xFFFFu;  // bit j: key j of the tile exists
    // Partial sums over 16 dims each, added pairwise: shorter chains round less
    // than one of 128 terms.
    float4_t part[D / 16];
#pragma unroll
    for (int i = 0; i < D / 16; i += 2) {
      part[i] = part[i + 1] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        part[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.k[i][s], qf[i][s], part[i], 0, 0, 0);
        part[i + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.k[i + 1][s], qf[i + 1][s], part[i + 1], 0, 0, 0);
      }
      part[i] += part[i + 1];
      if (i & 2) part[i - 2] += part[i];
      if (i == 6) part[0] += part[4];
    }
    const int32_t p0 = base + 16 * tile + 4 * grp;
    float s[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool vis = ((mapped >> (4 * grp + e)) & 1u) && p0 + e >= lo && p0 + e <= hi;
      s[e] = vis ? part[0][e] * a.scale_log2 : -INFINITY;
    }
    float bm = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
    bm = max_xor32_f(max_xor16_f(bm));
    const float mn = fmaxf(m, bm);
    const float alpha = mn == -INFINITY ? 1.f : exp2f(m - mn);
    float p[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = s[e] == -INFINITY ? 0.f : exp2f(s[e] - mn);
    l = l * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
    m = mn;
    // V rows that no column sees hold anything: zeros take their place. A
    // value that is not finite in a row that only some columns see must not
    // reach the others as 0 * inf: such a tile is multiplied column by column.
    float finite = 0.f;
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const bool here = (mapped >> (4 * grp + st)) & 1u;
#pragma unroll
      for (int j = 0; j < J; ++j) {
        if (!here) cur.v[st][j] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) finite = __builtin_fmaf(cur.v[st][j][c], 0.f, finite);
      }
    }
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[j][c] *= alpha;
    if (!__ballot(finite != finite)) {
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
          for (int c = 0; c < 4; ++c)
            acc[j][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.v[st][j][c], p[st], acc[j][c], 0, 0, 0);
    } else {
      for (int x = 0; x < 16; ++x) {
        const int32_t xlo = __shfl(lo, x, 64), xhi = __shfl(hi, x, 64);
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            float4_t sum = acc[j][c];
#pragma unroll
            for (int st = 0; st < 4; ++st) {
              const bool vis = p0 + st >= xlo && p0 + st <= xhi;
              sum = __builtin_amdgcn_mfma_f32_16x16x4f32(vis ? cur.v[st][j][c] : 0.f, p[st], sum, 0, 0, 0);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[j][c][e] = col == x ? sum[e] : acc[j][c][e];
          }
      }
    }
    cur = nxt;
  }
  // Merge the waves' states; a wave that saw no key holds (-inf, 0, 0).
  l = sum_xor32_f(sum_xor16_f(l));
  if (grp == 0) {
    msh[wave][col] = m;
    lsh[wave][col] = l;
  }
  __syncthreads();
  float most = -INFINITY;
#pragma unroll
  for (int w = 0; w < kTileWaves; ++w) most = fmaxf(most, msh[w][col]);
  const float weight = m == -INFINITY ? 0.f : exp2f(m - most);
  auto slice = [&](int half, int j, int e) {
    return reinterpret_cast<float4_t*>(&buf[half][col * kColStride + 64 * j + 16 * grp + 4 * e]);
  };
  constexpr int kHalf = kTileWaves / 2;
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[j][c] = weight == 0.f ? float4_t{0.f, 0.f, 0.f, 0.f} : acc[j][c] * weight;
  if (wave >= kHalf) {
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *slice(wave - kHalf, j, e) = float4_t{acc[j][0][e], acc[j][1][e], acc[j][2][e], acc[j][3][e]};
  }
  __syncthreads();
  if (wave < kHalf) {
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *slice(wave, j, e) += float4_t{acc[j][0][e], acc[j][1][e], acc[j][2][e], acc[j][3][e]};
  }
  __syncthreads();
  for (int i = tid; i < 16 * D / 4; i += 64 * kTileWaves) {
    const int x = i / (D / 4), d = 4 * (i % (D / 4));
    const int xg = x / T;
    const int64_t xt = t0 + x % T;
    if (xg >= G || xt >= qe) continue;
    float mx = -INFINITY, total = 0.f;
#pragma unroll
    for (int w = 0; w < kTileWaves; ++w) mx = fmaxf(mx, msh[w][x]);
#pragma unroll
    for (int w = 0; w < kTileWaves; ++w) total += msh[w][x] == -INFINITY ? 0.f : exp2f(msh[w][x] - mx) * lsh[w][x];
    float4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kHalf; ++w) o += *reinterpret_cast<const float4_t*>(&buf[w][x * kColStride + d]);
    const float inv = 1.f / total;  // an empty visible range gives 0 / 0 = NaN
    float* op = static_cast<float*>(a.out) + xt * a.o_s0 + (static_cast<int64_t>(h) * G + xg) * a.o_s1 + d * a.o_s2;
#pragma unroll
    for (int e = 0; e < 4; ++e) op[e * a.o_s2] = o[e] * inv;
  }
}

// What attention_f32_kernel assumes beyond the any-shape kernel: vector rows,
// positions and block sizes within 32 bits, a grid in range.
bool f32_tiles_supported(const AttnArgs& a) {
  const bool rows = a.q_s2 == 1 && a.q_s0 % 4 == 0 && a.q_s1 % 4 == 0 && aligned16(a.q) && a.c_s[4] == 1 &&
                    a.c_s[0] % 4 == 0 && a.c_s[1] % 4 == 0 && a.c_s[2] % 4 == 0 && a.c_s[3] % 4 == 0 && aligned16(a.cache);
  return a.mode == 0 && rows && (a.head_dim == 64 || a.head_dim == 128) && a.group <= 16 && a.num_requests > 0 &&
         a.num_blocks > 0 && a.block_size > 0 && a.width * a.block_size < (int64_t{1} << 30) &&
         a.num_tokens + a.num_requests < (int64_t{1} << 30);
}

int launch_f32_tiles(const AttnArgs& a, hipStream_t s) {
  const int32_t T = 16 / a.group;
  const int64_t slots = a.num_tokens / T + a.num_requests;
  const dim3 grid(static_cast<unsigned>(slots + (a.num_tokens + kTidyRows - 1) / kTidyRows),
                  static_cast<unsigned>(a.num_kv_heads));
  if (a.head_dim == 64) hipLaunchKernelGGL(attention_f32_kernel<64>, grid, dim3(64 * kTileWaves), 0, s, a, T, slots);
  else hipLaunchKernelGGL(attention_f32_kernel<128>, grid, dim3(64 * kTileWaves), 0, s, a, T, slots);
  MVLLM_LAUNCH_CHECK("attention_f32_kernel");
  return MVLLM_OK;
}

template <typename T, int DPL, int WAVES>
void launch_generic_w(const AttnArgs& a, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.num_tokens), static_cast<unsigned>(a.num_q_heads));
  hipLaunchKernelGGL((attention_generic_kernel<T, DPL, WAVES>), grid, dim3(64 * WAVES), 0, s, a);
}

template <typename T>
int launch_generic_t(const AttnArgs& a, int dpl, hipStream_t s) {
  const bool long_reach = a.width * a.block_size > 1024;
  switch (dpl) {
    case 1: long_reach ? launch_generic_w<T, 1, 16>(a, s) : launch_generic_w<T, 1, 4>(a, s); break;
    case 2: long_reach ? launch_generic_w<T, 2, 16>(a, s) : launch_generic_w<T, 2, 4>(a, s); break;
    case 4: long_reach ? launch_generic_w<T, 4, 8>(a, s) : launch_generic_w<T, 4, 4>(a, s); break;
    default: long_reach ? launch_generic_w<T, 8, 8>(a, s) : launch_generic_w<T, 8, 4>(a, s); break;
  }
  return MVLLM_OK;
}

}  // namespace

int launch_generic(const AttnArgs& a, int32_t dtype, hipStream_t s) {
  if (a.head_dim > 64 * kMaxDimPerLane)
    return fail(MVLLM_ERR_UNSUPPORTED, "head_dim %d exceeds %d", a.head_dim, 64 * kMaxDimPerLane);
  if (a.num_tokens == 0 || a.num_q_heads == 0) return MVLLM_OK;
  if (a.num_tokens > INT32_MAX || a.num_q_heads > 65535)
    return fail(MVLLM_ERR_INVALID, "generic attention grid too large");
  if (dtype == MVLLM_DTYPE_F32 && f32_tiles_supported(a)) return launch_f32_tiles(a, s);
  const int dpl = a.head_dim <= 64 ? 1 : a.head_dim <= 128 ? 2 : a.head_dim <= 256 ? 4 : 8;
  int rc = MVLLM_OK;
  switch (dtype) {
    case MVLLM_DTYPE_F32: rc = launch_generic_t<float>(a, dpl, s); break;
    case MVLLM_DTYPE_F16: rc = launch_generic_t<f16_t>(a, dpl, s); break;
    case MVLLM_DTYPE_BF16: rc = launch_generic_t<bf16_t>(a, dpl, s); break;
    default: return fail(MVLLM_ERR_UNSUPPORTED, "unsupported dtype code %d", dtype);
  }
  if (rc) return rc;
  MVLLM_LAUNCH_CHECK("attention_generic_kernel");
  return MVLLM_OK;
}

}  // namespace mvllm
