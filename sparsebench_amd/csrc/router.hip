// Router side of the MoE layer on gfx950: plain top-k and token rounding
// (the reference's sparsebench/token_rounding.py: top_k_assignments at
// 39-46, round_counts at 49-55, token_rounding at 58-81), with the rounding
// fused into routing: scores go in, and out come the assignment list and
// the block-sparse layout that SDD / DSD / the assigned combine consume,
// with no host sync (the reference needs one, for nonzero()).
//
// Token rounding, per expert e (f_e = its top-k count):
//   target_e = f_e rounded to the nearest multiple of the tile, ties down,
//              at most floor(T / tile) * tile;
//   keep (t, e) for the target_e best tokens of column e, where picks keep
//   their score s and the others rank at s - 1, ties going to the lower
//   token (the reference's stable descending sort);
//   weight (t, e) = s[t, e] / sum of s over t's kept experts, the sum taken
//   in ascending expert order.
// The list is in (token, expert) order, like the reference's nonzero().
//
// Launches:
//   1. topk      one lane per token (one wave per token when E x k is
//                large): the k best experts (value, then lower index),
//                per-chunk pick counts, the shifted scores stored
//                expert-major, and (for top_k_assignments) the list itself.
//   2. targets   one workgroup: counts -> targets -> padded_offsets.
//   3. select    one workgroup per expert: radix select (4 passes of 8 bits)
//                of the target-th largest shifted score, then the keep
//                bitmask, its per-word prefix counts and row_token.
//   4. emit      one workgroup per 32 tokens (a word of every expert's
//                bitmask): kept counts and score totals, token_offsets,
//                token / expert / weight / copy_row; the other workgroups
//                write row_offsets, col_indices, row_block_expert, -1 rows.

#include "common.hpp"
#include "expert_chunks.hpp"
#include "layout.hpp"

namespace sb {
namespace {

constexpr int kTopkTokensPerGroup = 64;  // 4 waves x 16 tokens
constexpr int kTopkThreads = 256;
constexpr int kMaxPerLane = kMaxExperts / 64;
constexpr int kSelectThreads = 1024;
constexpr int kEmitThreads = 256;
constexpr int kEmitWaves = kEmitThreads / 64;

// Order-preserving map of a float to uint32 (larger float -> larger key).
// -0 counts as +0 and every NaN as the largest value, as in a sort that
// compares values.
__device__ __forceinline__ uint32_t sort_key(float f) {
  if (f == 0.0f) f = 0.0f;
  uint32_t u = __float_as_uint(f);
  if (f != f) u = 0x7fc00000u;
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Better of two (score, expert) candidates: higher score, then lower index.
__device__ __forceinline__ bool better(float a, int ia, float b, int ib) {
  return a > b || (a == b && ia < ib);
}

template <int PER>
__global__ void __launch_bounds__(kTopkThreads)
    router_topk_kernel(const float* __restrict__ scores, int64_t num_tokens, int32_t num_experts, int32_t k,
                       float* __restrict__ shifted, int32_t* __restrict__ chunk_counts,
                       int32_t* __restrict__ top_idx, float* __restrict__ top_weight) {
  // With E <= 256 the shifted scores go through an LDS tile [E][64 tokens]
  // so that the expert-major stores are 64-token rows, not scattered words.
  constexpr bool kTile = PER <= 4;
  constexpr int kTileStride = kTopkTokensPerGroup + 1;
  constexpr int kPerWave = kTopkTokensPerGroup / 4;
  // Tokens whose scores are loaded together (all loads in flight at once).
  constexpr int kBatch = PER <= 2 ? kPerWave : PER <= 4 ? 8 : 4;
  __shared__ int32_t hist[kMaxExperts];
  __shared__ float tile[kTile ? 64 * PER * kTileStride : 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (chunk_counts != nullptr)
    for (int e = tid; e < num_experts; e += kTopkThreads) hist[e] = 0;
  __syncthreads();

  const int64_t group_base = static_cast<int64_t>(blockIdx.x) * kTopkTokensPerGroup;
  for (int j0 = 0; j0 < kPerWave; j0 += kBatch) {
    float vb[kBatch][PER];
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      const int64_t t = group_base + wave * kPerWave + j0 + b;
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int e = lane + 64 * i;
        vb[b][i] = (t < num_tokens && e < num_experts) ? scores[t * num_experts + e] : 0.0f;
      }
    }
    // The k rounds of all kBatch tokens in lockstep: their shuffle chains
    // are independent, so they overlap instead of running one after another.
    uint32_t picked[kBatch];
    float total[kBatch];
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      picked[b] = 0;
      total[b] = 0.0f;
    }
    for (int r = 0; r < k; ++r) {
      float bv[kBatch];
      int bi[kBatch];
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        bv[b] = 0.0f;
        bi[b] = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          const int e = lane + 64 * i;
          if (e < num_experts && !((picked[b] >> i) & 1u) && (bi[b] == 0x7fffffff || better(vb[b][i], e, bv[b], bi[b]))) {
            bv[b] = vb[b][i];
            bi[b] = e;
          }
        }
      }
      for (int d = 32; d >= 1; d >>= 1) {
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
          const float ov = __shfl_xor(bv[b], d, 64);
          const int oi = __shfl_xor(bi[b], d, 64);
          if (oi != 0x7fffffff && (bi[b] == 0x7fffffff || better(ov, oi, bv[b], bi[b]))) {
            bv[b] = ov;
            bi[b] = oi;
          }
        }
      }
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        // bi[b]: the r-th best expert of token b, the same in every lane.
        if ((bi[b] & 63) == lane) picked[b] |= 1u << (bi[b] >> 6);
        total[b] += bv[b];  // in pick order, as a sum over the k picks
        const int64_t t = group_base + wave * kPerWave + j0 + b;
        if (lane == 0 && t < num_tokens) {
          if (top_idx != nullptr) top_idx[t * k + r] = bi[b];
          if (top_weight != nullptr) top_weight[t * k + r] = bv[b];  // raw score; normalized below
        }
      }
    }
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      const int t_local = wave * kPerWave + j0 + b;
      const int64_t t = group_base + t_local;
      if (t >= num_tokens) break;
      // Weights: the picked scores over their sum (lane 0 reads back what it wrote).
      if (top_weight != nullptr && lane == 0)
        for (int r = 0; r < k; ++r) top_weight[t * k + r] = top_weight[t * k + r] / total[b];
      if (shifted != nullptr) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          const int e = lane + 64 * i;
          if (e < num_experts) {
            const float sv = ((picked[b] >> i) & 1u) ? vb[b][i] : vb[b][i] - 1.0f;
            if constexpr (kTile) tile[e * kTileStride + t_local] = sv;
            else shifted[static_cast<int64_t>(e) * num_tokens + t] = sv;
          }
        }
      }
      if (chunk_counts != nullptr) {
#pragma unroll
        for (int i = 0; i < PER; ++i)
          if ((picked[b] >> i) & 1u) atomicAdd(&hist[lane + 64 * i], 1);
      }
    }
  }
  __syncthreads();
  if constexpr (kTile) {
    if (shifted != nullptr) {
      for (int i = tid; i < num_experts * kTopkTokensPerGroup; i += kTopkThreads) {
        const int e = i / kTopkTokensPerGroup, tl = i % kTopkTokensPerGroup;
        const int64_t t = group_base + tl;
        if (t < num_tokens) shifted[static_cast<int64_t>(e) * num_tokens + t] = tile[e * kTileStride + tl];
      }
    }
  }
  if (chunk_counts != nullptr)
    for (int e = tid; e < num_experts; e += kTopkThreads)
      chunk_counts[static_cast<int64_t>(blockIdx.x) * num_experts + e] = hist[e];
}

// A lane's KMAX best (score, expert), sorted by (score desc, expert asc), of
// which the first k are kept.
template <int KMAX>
struct BestK {
  float bv[KMAX];
  int bi[KMAX];
  int k;
  __device__ __forceinline__ explicit BestK(int kept) : k(kept) {
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
      bv[j] = 0.0f;
      bi[j] = 0x7fffffff;  // empty
    }
  }
  __device__ __forceinline__ void offer(float v, int e) {
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {  // selects, not branches: the lanes disagree at every step
      const bool in = (j < k) & ((bi[j] == 0x7fffffff) | (v > bv[j]) | ((v == bv[j]) & (e < bi[j])));
      const float tv = in ? bv[j] : v;
      const int ti = in ? bi[j] : e;
      bv[j] = in ? v : bv[j];
      bi[j] = in ? e : bi[j];
      v = tv;
      e = ti;
    }
  }
};

// Top-k with one lane per token (64 tokens per workgroup, the same chunking
// as router_topk_kernel). The workgroup's four waves read the scores a tile of
// 64 tokens x up to kLaneTile experts at a time into LDS, whole rows of a
// token side by side, and write the shifted scores from there; the first
// wave's lanes walk their tokens' rows in the tile in expert order and keep
// the KMAX best in registers (BestK): each new (score, e) is bubbled in with
// compare-and-swap steps, so an equal score behind an earlier expert stays
// behind it. No lane talks to another, and the
// expert-major stores of the shifted scores are 64 consecutive tokens per
// instruction. The outputs are those of router_topk_kernel. Bound by the
// latency of its loads: with each lane reading its own row from memory,
// twice, 13.6 us at T = 4096, E = 64, k = 2; this takes 8.3.
constexpr int kLaneTile = 128;

template <int KMAX>
__global__ void __launch_bounds__(kTopkThreads)
    router_topk_lane_kernel(const float* __restrict__ scores, int64_t num_tokens, int32_t num_experts, int32_t k,
                            float* __restrict__ shifted, int32_t* __restrict__ chunk_counts,
                            int32_t* __restrict__ top_idx, float* __restrict__ top_weight) {
  __shared__ int32_t hist[kMaxExperts];
  __shared__ uint32_t picked_bits[64 * (kMaxExperts / 32)];  // lane-major: this lane's picks, one bit per expert
  __shared__ float tile[64 * (kLaneTile + 1)];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int words = (num_experts + 31) / 32;
  if (chunk_counts != nullptr)
    for (int e = tid; e < num_experts; e += kTopkThreads) hist[e] = 0;
  for (int w = tid; w < 64 * words; w += kTopkThreads) picked_bits[w] = 0u;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * 64;
  const int64_t t = t0 + lane;
  const int tokens = static_cast<int>(min(num_tokens - t0, int64_t{64}));
  // Experts e0 .. e0+width of the workgroup's tokens; synchronizes around it.
  auto load_tile = [&](int e0, int width) {
    constexpr int kRows = 64 / (kTopkThreads / 64);  // tokens of a wave, all their loads in flight together
    float v[kRows][kLaneTile / 64];
#pragma unroll
    for (int r = 0; r < kRows; ++r)
#pragma unroll
      for (int c = 0; c < kLaneTile / 64; ++c) {
        const int tl = wave * kRows + r, e = 64 * c + lane;
        // Past the tile: the last token or expert again (a load of its own
        // branch for each would wait for the one before).
        v[r][c] = scores[(t0 + min(tl, tokens - 1)) * num_experts + e0 + min(e, width - 1)];
      }
    __syncthreads();  // the tile before has been read
#pragma unroll
    for (int r = 0; r < kRows; ++r)
#pragma unroll
      for (int c = 0; c < kLaneTile / 64; ++c)
        tile[(wave * kRows + r) * (kLaneTile + 1) + 64 * c + lane] = v[r][c];
    __syncthreads();
  };

  BestK<KMAX> best(k);
  for (int e0 = 0; e0 < num_experts; e0 += kLaneTile) {
    const int width = min(kLaneTile, num_experts - e0);
    load_tile(e0, width);
    if (wave == 0 && lane < tokens) {
      constexpr int kBatch = 16;  // LDS reads in flight
      int e = 0;
      for (; e + kBatch <= width; e += kBatch) {
        float v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) v[u] = tile[lane * (kLaneTile + 1) + e + u];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) best.offer(v[u], e0 + e + u);
      }
      for (; e < width; ++e) best.offer(tile[lane * (kLaneTile + 1) + e], e0 + e);
    }
  }
  if (wave == 0 && lane < tokens) {
    float total = 0.0f;
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
      if (j < k && best.bi[j] != 0x7fffffff) {
        total += best.bv[j];  // in pick order
        picked_bits[lane * words + (best.bi[j] >> 5)] |= 1u << (best.bi[j] & 31);
        if (chunk_counts != nullptr) atomicAdd(&hist[best.bi[j]], 1);
        if (top_idx != nullptr) top_idx[t * k + j] = best.bi[j];
      }
    }
    if (top_weight != nullptr)
#pragma unroll
      for (int j = 0; j < KMAX; ++j)
        if (j < k) top_weight[t * k + j] = best.bv[j] / total;
  }
  __syncthreads();
  if (shifted != nullptr) {
    for (int e0 = 0; e0 < num_experts; e0 += kLaneTile) {
      const int width = min(kLaneTile, num_experts - e0);
      if (num_experts > kLaneTile) load_tile(e0, width);  // else the tile still holds all of them
      if (lane < tokens)
        for (int e = wave; e < width; e += kTopkThreads / 64) {
          const float v = tile[lane * (kLaneTile + 1) + e];
          const bool pick = (picked_bits[lane * words + ((e0 + e) >> 5)] >> ((e0 + e) & 31)) & 1u;
          shifted[static_cast<int64_t>(e0 + e) * num_tokens + t] = pick ? v : v - 1.0f;
        }
    }
  }
  if (chunk_counts != nullptr)
    for (int e = tid; e < num_experts; e += kTopkThreads)
      chunk_counts[static_cast<int64_t>(blockIdx.x) * num_experts + e] = hist[e];
}

// Top-k alone, each lane walking its token's own row from memory: for few
// experts, whose rows the tiles' loads would leave mostly idle, and for so many
// tokens that the waves hide the loads' latency, where the tiles' LDS keeps all
// but a few waves off a CU. The outputs are those of router_topk_kernel.
template <int KMAX>
__global__ void __launch_bounds__(64)
    router_topk_direct_kernel(const float* __restrict__ scores, int64_t num_tokens, int32_t num_experts, int32_t k,
                              int32_t* __restrict__ top_idx, float* __restrict__ top_weight) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 64 + threadIdx.x;
  if (t >= num_tokens) return;
  const float* row = scores + t * num_experts;
  BestK<KMAX> best(k);
  int e = 0;
  if ((num_experts & 3) == 0 && (reinterpret_cast<uintptr_t>(scores) & 15) == 0) {
    for (; e + 16 <= num_experts; e += 16) {  // 16 scores (four 16-byte loads) in flight
      float4 q[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) q[u] = *reinterpret_cast<const float4*>(row + e + 4 * u);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        best.offer(q[u].x, e + 4 * u);
        best.offer(q[u].y, e + 4 * u + 1);
        best.offer(q[u].z, e + 4 * u + 2);
        best.offer(q[u].w, e + 4 * u + 3);
      }
    }
    for (; e < num_experts; e += 4) {
      const float4 q = *reinterpret_cast<const float4*>(row + e);
      best.offer(q.x, e);
      best.offer(q.y, e + 1);
      best.offer(q.z, e + 2);
      best.offer(q.w, e + 3);
    }
  }
  for (; e < num_experts; ++e) best.offer(row[e], e);
  float total = 0.0f;
#pragma unroll
  for (int j = 0; j < KMAX; ++j)
    if (j < k) {
      if (top_idx != nullptr) top_idx[t * k + j] = best.bi[j];
      total += best.bv[j];  // in pick order
    }
  if (top_weight != nullptr)
#pragma unroll
    for (int j = 0; j < KMAX; ++j)
      if (j < k) top_weight[t * k + j] = best.bv[j] / total;
}

// Inclusive scan over the lanes of one 1024-lane workgroup.
__device__ __forceinline__ int32_t block_scan_1024(int32_t v, int32_t* wave_sums, int32_t* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = wave_inclusive_scan(v);
  if (lane == 63) wave_sums[wave] = v;
  __syncthreads();
  int32_t before = 0, all = 0;
  for (int w = 0; w < 16; ++w) {
    if (w < wave) before += wave_sums[w];
    all += wave_sums[w];
  }
  __syncthreads();
  *total = all;
  return v + before;
}

__global__ void __launch_bounds__(1024)
    router_targets_kernel(const int32_t* __restrict__ chunk_counts, int32_t num_chunks, int32_t num_experts,
                          int64_t num_tokens, int32_t tile, int32_t block_size, int32_t* __restrict__ target,
                          int32_t* __restrict__ padded_offsets, int32_t* __restrict__ error) {
  __shared__ int32_t counts[kMaxExperts];
  __shared__ int32_t wave_sums[16];
  const int tid = threadIdx.x;
  for (int e = tid; e < num_experts; e += 1024) counts[e] = 0;
  __syncthreads();
  // Column sums of chunk_counts [chunks, E], read in order, 8 loads in flight per lane.
  constexpr int kPer = 8;
  const int64_t total_items = static_cast<int64_t>(num_chunks) * num_experts;
  for (int64_t base = 0; base < total_items; base += 1024 * kPer) {
    int32_t v[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int64_t i = base + u * 1024 + tid;
      v[u] = i < total_items ? chunk_counts[i] : 0;
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u)
      if (v[u] != 0) atomicAdd(&counts[(base + u * 1024 + tid) % num_experts], v[u]);
  }
  __syncthreads();
  int32_t padded = 0;
  if (tid < num_experts) {
    const int32_t f = counts[tid];
    const int32_t low = f / tile * tile;
    const int32_t high = low + (f % tile > 0 ? tile : 0);
    int32_t rounded = (high - f < f - low) ? high : low;  // nearest, ties down
    const int64_t cap = num_tokens / tile * tile;
    if (rounded > cap) rounded = static_cast<int32_t>(cap);
    target[tid] = rounded;
    padded = (rounded + block_size - 1) / block_size * block_size;
  }
  int32_t total;
  const int32_t incl = block_scan_1024(padded, wave_sums, &total);
  if (tid < num_experts) padded_offsets[tid + 1] = incl;
  if (tid == 0) {
    padded_offsets[0] = 0;
    error[0] = 0;
  }
}

__device__ __forceinline__ uint64_t lanes_below() {
  const int lane = threadIdx.x & 63;
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// hist[bin] += 1 for every active lane, one LDS atomic per distinct bin in
// the wave (lanes with the same bin found by one ballot per bin bit).
// Softmax scores share few top-byte values, so plain per-lane atomics
// would pile onto one or two addresses.
__device__ __forceinline__ void wave_hist_add(int32_t* hist, uint32_t bin, bool active) {
  uint64_t peers = __ballot(active);
  if (peers == 0) return;  // after the first pass or two, most waves
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const bool bit = (bin >> b) & 1u;
    const uint64_t ones = __ballot(active && bit);
    peers &= bit ? ones : ~ones;
  }
  if (active && (peers & lanes_below()) == 0) atomicAdd(&hist[bin], __popcll(peers));
}

constexpr int kSelectLdsTokens = 32768;  // a column of up to this many keys stays in LDS (128 KB)

// One workgroup per expert e: which tokens it keeps, and their rows.
__global__ void __launch_bounds__(kSelectThreads)
    router_select_kernel(const float* __restrict__ shifted, int64_t num_tokens, const int32_t* __restrict__ target,
                         const int32_t* __restrict__ padded_offsets, uint32_t* __restrict__ keep_mask,
                         int32_t* __restrict__ keep_prefix, int32_t* __restrict__ row_token) {
  __shared__ uint32_t keys[kSelectLdsTokens];
  __shared__ int32_t hist[4][256];  // of each pass
  __shared__ int32_t wave_sums[16];
  __shared__ uint32_t s_prefix, s_prefix_mask;
  __shared__ bool s_done;
  __shared__ int32_t s_remaining;
  __shared__ uint32_t counts[kSelectLdsTokens / 64];
  const int tid = threadIdx.x;
  const int e = blockIdx.x;
  const float* col = shifted + static_cast<int64_t>(e) * num_tokens;
  const int32_t tgt = target[e];
  const int64_t words = (num_tokens + 31) / 32;
  uint32_t* mask = keep_mask + static_cast<int64_t>(e) * words;
  int32_t* pref = keep_prefix + static_cast<int64_t>(e) * words;

  // Keys of the column, computed once (in LDS when they fit).
  const bool in_lds = num_tokens <= kSelectLdsTokens;
  if (in_lds) {
    constexpr int kPer = 8;
    for (int64_t base = 0; base < num_tokens; base += kSelectThreads * kPer) {
      float v[kPer];
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int64_t t = base + u * kSelectThreads + tid;
        v[u] = col[min(t, num_tokens - 1)];
      }
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int64_t t = base + u * kSelectThreads + tid;
        if (t < num_tokens) keys[t] = sort_key(v[u]);
      }
    }
    __syncthreads();
  }
  auto key_at = [&](int64_t t) -> uint32_t { return in_lds ? keys[t] : sort_key(col[t]); };

  // Keep t iff key > thr, or key == thr and fewer than `ties` tokens before it
  // have that key.
  uint32_t thr = 0;
  int32_t ties = 0;
  bool keep_all = false, keep_none = false;
  if (tgt <= 0) {
    keep_none = true;
  } else if (tgt >= num_tokens) {
    keep_all = true;
  } else {
    if (tid == 0) {
      s_prefix = 0;
      s_prefix_mask = 0;
      s_remaining = tgt;
      s_done = false;
    }
    static_assert(kSelectThreads == 4 * 256, "one lane a bin of every pass");
    hist[tid >> 8][tid & 255] = 0;
    __syncthreads();
    for (int pass = 0; pass < 4; ++pass) {
      const int shift = 24 - 8 * pass;
      const uint32_t pre = s_prefix, pmask = s_prefix_mask;
      for (int64_t base = 0; base < num_tokens; base += kSelectThreads) {  // same trip count in every lane
        const int64_t t = base + tid;
        const uint32_t key = t < num_tokens ? key_at(t) : 0u;
        wave_hist_add(hist[pass], (key >> shift) & 255u, t < num_tokens && (key & pmask) == pre);
      }
      __syncthreads();
      if (tid < 64) {
        // Wave 0: lane l holds bins 255-4l .. 252-4l (descending). A suffix
        // count from the top finds the bin where the rem-th largest falls.
        const int32_t rem = s_remaining;
        int32_t c[4], own = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          c[q] = hist[pass][255 - 4 * tid - q];
          own += c[q];
        }
        const int32_t incl = wave_inclusive_scan(own);  // keys in bins above and including this lane's four
        int32_t above = incl - own;  // keys in higher bins than this lane's
        // The lane whose four bins reach rem: the first with incl >= rem.
        const uint64_t reach = __ballot(incl >= rem);
        if (reach != 0 && tid == __builtin_ctzll(reach)) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (above + c[q] >= rem) {
              const uint32_t found = pre | (static_cast<uint32_t>(255 - 4 * tid - q) << shift);
              // All of the bin's keys are kept: keep every key above found - 1.
              s_done = above + c[q] == rem && found != 0;
              s_prefix = s_done ? found - 1 : found;
              s_prefix_mask = pmask | (255u << shift);
              s_remaining = s_done ? 0 : rem - above;
              break;
            }
            above += c[q];
          }
        }
      }
      __syncthreads();
      if (s_done) break;
    }
    thr = s_prefix;
    ties = s_remaining;  // keys == thr to keep, in token order
  }

  // Keep bitmask, 64 tokens a wave by ballot. The counts above and at the
  // threshold of every 64 tokens of a round are scanned together (two halves
  // of one word, each at most kSelectLdsTokens); a token's rank among the
  // kept, its expert's row, follows from them.
  constexpr int kRoundWaves = kSelectLdsTokens / 64;
  static_assert(kRoundWaves <= kSelectThreads && kSelectLdsTokens < 65536, "one scan a round, two 16-bit counts");
  const int lane = tid & 63, wave = tid >> 6;
  const int32_t row0 = padded_offsets[e];
  auto masks = [&](int64_t t, uint64_t* above, uint64_t* at) {
    const bool in = t < num_tokens && !keep_none;
    const uint32_t key = in && !keep_all ? key_at(t) : 0u;
    *above = __ballot(in && (keep_all || key > thr));
    *at = __ballot(in && !keep_all && key == thr);
  };
  int32_t above_before = 0, at_before = 0;  // of earlier rounds
  for (int64_t base = 0; base < num_tokens; base += kSelectLdsTokens) {
    const int waves = static_cast<int>(min((num_tokens - base + 63) / 64, static_cast<int64_t>(kRoundWaves)));
    for (int w = wave; w < waves; w += kSelectThreads / 64) {
      uint64_t above, at;
      masks(base + 64 * w + lane, &above, &at);
      if (lane == 0) counts[w] = (static_cast<uint32_t>(__popcll(above)) << 16) + __popcll(at);
    }
    __syncthreads();
    int32_t total;
    const int32_t mine = tid < waves ? static_cast<int32_t>(counts[tid]) : 0;
    const int32_t incl = block_scan_1024(mine, wave_sums, &total);  // synchronizes the workgroup
    if (tid < waves) counts[tid] = static_cast<uint32_t>(incl - mine);
    __syncthreads();
    for (int w = wave; w < waves; w += kSelectThreads / 64) {
      const int64_t t = base + 64 * w + lane;
      uint64_t above, at;
      masks(t, &above, &at);
      const int32_t tied = at_before + static_cast<int32_t>(counts[w] & 0xffffu);  // ties before these 64
      const bool keep = ((above >> lane) & 1u) ||
                        (((at >> lane) & 1u) && tied + __popcll(at & lanes_below()) < ties);
      const uint64_t kept = __ballot(keep);
      const int32_t first = above_before + static_cast<int32_t>(counts[w] >> 16) + min(tied, ties);
      if (keep) row_token[row0 + first + __popcll(kept & lanes_below())] = static_cast<int32_t>(t);
      const int64_t word = t / 32;
      if ((lane & 31) == 0 && word < words) {
        mask[word] = static_cast<uint32_t>(kept >> lane);
        pref[word] = first + (lane == 0 ? 0 : __popc(static_cast<uint32_t>(kept)));
      }
    }
    above_before += static_cast<int32_t>(static_cast<uint32_t>(total) >> 16);
    at_before += total & 0xffff;
    __syncthreads();
  }
}

// Workgroup w < words: tokens 32 w .. 32 w + 31, one word of every expert's
// keep bitmask. The copies of earlier tokens are the experts' prefix counts
// at that word, so the workgroup finds its place in the list by itself; each
// of its waves takes 8 tokens, a lane per expert: kept count, score total
// (added in ascending expert order), then the token's entries in expert order.
// The capacity past the list's end is filled with -1 / -1 / 0 / -1. The
// workgroups past the words write the block-sparse layout. (Separate kernels
// for counts, their scan, the list and the layout took 4.7 + 5.4 + 4.7 + 4.6
// us at T = 4096, E = 64, each little more than its launch; this takes
// 6.1. The whole rounding at T = 4096, before and now: E = 300, k = 4 137 and 84
// us; E = 512, k = 8 232 and 167; E = 1000, k = 8 338 and 301.)
template <int PER>
__global__ void __launch_bounds__(kEmitThreads)
    router_emit_kernel(const float* __restrict__ scores, int64_t num_tokens, int32_t num_experts,
                       const uint32_t* __restrict__ keep_mask, const int32_t* __restrict__ keep_prefix,
                       const int32_t* __restrict__ tokens_per_expert, const int32_t* __restrict__ padded_offsets,
                       int64_t capacity, int32_t block_size, int32_t ffn_blocks, int32_t max_row_blocks,
                       int64_t max_rows, int32_t* __restrict__ token_offsets, int32_t* __restrict__ num_assignments,
                       int32_t* __restrict__ token_of_copy, int32_t* __restrict__ expert_of_copy,
                       float* __restrict__ weight_of_copy, int32_t* __restrict__ copy_row,
                       int32_t* __restrict__ row_token, int32_t* __restrict__ row_block_expert,
                       int32_t* __restrict__ row_offsets, int32_t* __restrict__ col_indices) {
  constexpr int kPerWave = 32 / kEmitWaves;
  __shared__ int32_t lds[2 * kMaxExperts + 1];
  __shared__ int32_t sums[2][kEmitWaves];
  __shared__ int32_t cnt[32];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t words = (num_tokens + 31) / 32;
  const int64_t word = blockIdx.x;
  if (word >= words) {
    int32_t* offs = lds;
    int32_t* cnts = lds + kMaxExperts + 1;
    for (int e = tid; e <= num_experts; e += kEmitThreads) offs[e] = padded_offsets[e];
    for (int e = tid; e < num_experts; e += kEmitThreads) cnts[e] = tokens_per_expert[e];
    __syncthreads();
    layout_item((word - words) * kEmitThreads + tid, offs, cnts, num_experts, block_size, ffn_blocks, max_row_blocks,
                max_rows, row_token, row_block_expert, row_offsets, col_indices);
    return;
  }
  // The wave's tokens' scores, lane l the experts l, l + 64, ...: read whole,
  // ahead of the bitmasks, so that their loads wait together.
  float s[kPerWave][PER];
#pragma unroll
  for (int j = 0; j < kPerWave; ++j)
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int64_t t = min(word * 32 + wave * kPerWave + j, num_tokens - 1);
      s[j][i] = scores[t * num_experts + min(64 * i + lane, num_experts - 1)];  // unused past the tokens and experts
    }
  uint32_t* mask = reinterpret_cast<uint32_t*>(lds);  // [E] this word of the experts' bitmasks
  int32_t* row0 = lds + kMaxExperts;                  // [E] row of the expert's first kept token of the word
  int32_t before = 0, all = 0;  // copies of earlier tokens, and of all
  for (int e = tid; e < num_experts; e += kEmitThreads) {
    const int64_t at = static_cast<int64_t>(e) * words + word;
    const int32_t prefix = keep_prefix[at];
    mask[e] = keep_mask[at];
    row0[e] = padded_offsets[e] + prefix;
    before += prefix;
    all += tokens_per_expert[e];
  }
  before = wave_inclusive_scan_total(before);
  all = wave_inclusive_scan_total(all);
  if (lane == 0) {
    sums[0][wave] = before;
    sums[1][wave] = all;
  }
  __syncthreads();
  before = all = 0;
  for (int w = 0; w < kEmitWaves; ++w) {
    before += sums[0][w];
    all += sums[1][w];
  }

  float total[kPerWave];
#pragma unroll
  for (int j = 0; j < kPerWave; ++j) {
    const int b = wave * kPerWave + j;
    int32_t n = 0;
    total[j] = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = 64 * i + lane;
      uint64_t bal = __ballot(e < num_experts && ((mask[e] >> b) & 1u));  // never set past the tokens
      n += __popcll(bal);
      while (bal != 0) {  // sequential, in expert order
        const int l = __builtin_ctzll(bal);
        bal &= bal - 1;
        total[j] += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s[j][i]), l));
      }
    }
    if (lane == 0) cnt[b] = n;
  }
  __syncthreads();
  const int32_t own = lane < 32 ? cnt[lane] : 0;
  const int32_t first = before + wave_inclusive_scan(own) - own;  // lane b < 32: where token b's entries start
  if (wave == 0 && lane < 32 && word * 32 + lane < num_tokens) token_offsets[word * 32 + lane] = first;
  if (word == words - 1 && tid == 0) {
    token_offsets[num_tokens] = all;
    num_assignments[0] = all;
  }
#pragma unroll
  for (int j = 0; j < kPerWave; ++j) {
    const int b = wave * kPerWave + j;
    const int64_t t = word * 32 + b;
    int32_t c = __builtin_amdgcn_readlane(first, b);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = 64 * i + lane;
      const bool keep = e < num_experts && ((mask[e] >> b) & 1u);
      const uint64_t bal = __ballot(keep);
      if (keep) {
        const int64_t slot = c + __popcll(bal & lanes_below());
        token_of_copy[slot] = static_cast<int32_t>(t);
        expert_of_copy[slot] = e;
        weight_of_copy[slot] = s[j][i] / total[j];
        copy_row[slot] = row0[e] + __popc(mask[e] & ((1u << b) - 1u));
      }
      c += __popcll(bal);
    }
  }
  for (int64_t i = all + word * kEmitThreads + tid; i < capacity; i += words * kEmitThreads) {
    token_of_copy[i] = -1;
    expert_of_copy[i] = -1;
    weight_of_copy[i] = 0.0f;
    copy_row[i] = -1;
  }
}

struct RouterSizes {
  int64_t max_assignments, workspace_elems, max_row_blocks, max_rows;
  int64_t chunks, words;
};

int router_sizes(int64_t num_tokens, int32_t num_experts, int32_t k, int32_t tile, int32_t block_size,
                 int32_t ffn_dim, RouterSizes* out) {
  constexpr int64_t kI32Max = 2147483647;
  if (num_tokens <= 0 || num_tokens > kI32Max / 2) return fail(SB_ERR_INVALID, "scores must be [T, E] with T > 0");
  if (num_experts <= 0 || num_experts > kMaxExperts)
    return fail(SB_ERR_INVALID, "num_experts must be in [1, %d], got %d", kMaxExperts, num_experts);
  if (k <= 0 || k > num_experts || k > 16)
    return fail(SB_ERR_INVALID, "k must be in [1, min(E, 16)], got %d", k);
  if (tile <= 0) return fail(SB_ERR_INVALID, "tile must be positive");
  // Rounding moves an expert by less than half a tile upwards.
  const int64_t cap = std::min<int64_t>(num_tokens * num_experts,
                                        num_tokens * k + static_cast<int64_t>(num_experts) * (tile / 2));
  int64_t rb = 0, rows = 0, ws_route = 0;
  if (int rc = sb_routing_sizes(cap, num_experts, ffn_dim, block_size, &rb, &rows, &ws_route)) return rc;
  out->max_assignments = cap;
  out->max_row_blocks = rb;
  out->max_rows = rows;
  out->chunks = (num_tokens + kTopkTokensPerGroup - 1) / kTopkTokensPerGroup;
  out->words = (num_tokens + 31) / 32;
  // chunk counts, shifted scores, keep mask, keep prefix; E + 2T words of the
  // size that callers are told are spare
  out->workspace_elems = out->chunks * num_experts + num_experts + num_tokens * num_experts +
                         2 * out->words * num_experts + 2 * num_tokens;
  return SB_OK;
}

int launch_topk(const float* scores, int64_t num_tokens, int32_t num_experts, int32_t k, float* shifted,
                int32_t* chunk_counts, int32_t* top_idx, float* top_weight, hipStream_t s) {
  const uint32_t groups = static_cast<uint32_t>((num_tokens + kTopkTokensPerGroup - 1) / kTopkTokensPerGroup);
  const int per = (num_experts + 63) / 64;
  // A lane per token unless its insertion work (E x the rounded-up k) is
  // large (4096 tokens, lane against wave form: E = 1000, k = 8 199 against
  // 239 us; E = 512, k = 16 253 against 339; E = 1000, k = 16 491 against
  // 472); the test hook SB_HOOK_TOPK_KERNEL = 1 forces the wave form, 2
  // the lane form.
  const int kmax = k <= 1 ? 1 : k <= 2 ? 2 : k <= 4 ? 4 : k <= 8 ? 8 : 16;
  const int forced = test_hook(SB_HOOK_TOPK_KERNEL);
  if (forced == 2 || (forced != 1 && kmax * num_experts <= 8192)) {
    // Alone, the direct form where a row takes few loads of 16 bytes and little
    // work (T = 4096, direct against tiles: E = 8, k = 2 2.8 and 3.8 us; E = 16,
    // k = 2 3.0 and 4.0; E = 60, k = 4 8.4 and 10.2; but E = 128, k = 8 31.8 and
    // 30.1; rows read 4 bytes at a time E = 33, k = 2 6.0 and 4.9) and from 512
    // groups on (T = 131072, E = 32, k = 2 5.5 and 13.1), there of rows that are
    // not whole 16 bytes only short ones (T = 300000, E = 129, k = 4 650 and 124).
    const bool wide = num_experts % 4 == 0 && aligned16(scores);
    const bool direct = shifted == nullptr && chunk_counts == nullptr &&
                        (num_experts <= 8 || (wide && kmax * num_experts <= 256) ||
                         (groups > 512 && (wide || num_experts <= std::max(48, 8 * kmax))));
    // Rows read 4 bytes at a time are read again and again from L1, which holds
    // those of a few waves: LDS that the kernel does not use keeps a CU at 13
    // (T = 300000, E = 45, k = 8 165 us without, 88 with).
    const uint32_t waves_lds = wide || num_experts <= 8 ? 0 : 12 * 1024;
#define SB_TOPK_LANE(K)                                                                                             \
  if (direct) router_topk_direct_kernel<K><<<groups, 64, waves_lds, s>>>(scores, num_tokens, num_experts, k, top_idx, top_weight); \
  else \
  router_topk_lane_kernel<K><<<groups, kTopkThreads, 0, s>>>(scores, num_tokens, num_experts, k, shifted, chunk_counts, top_idx, top_weight)
    if (k <= 1) { SB_TOPK_LANE(1); }
    else if (k <= 2) { SB_TOPK_LANE(2); }
    else if (k <= 4) { SB_TOPK_LANE(4); }
    else if (k <= 8) { SB_TOPK_LANE(8); }
    else { SB_TOPK_LANE(16); }
#undef SB_TOPK_LANE
    return check_launch("router top-k");
  }
#define SB_TOPK(P)                                                                                          \
  router_topk_kernel<P><<<groups, kTopkThreads, 0, s>>>(scores, num_tokens, num_experts, k, shifted, chunk_counts, \
                                                        top_idx, top_weight)
  if (per <= 1) SB_TOPK(1);
  else if (per <= 2) SB_TOPK(2);
  else if (per <= 4) SB_TOPK(4);
  else if (per <= 8) SB_TOPK(8);
  else SB_TOPK(kMaxPerLane);
#undef SB_TOPK
  return check_launch("router top-k");
}

}  // namespace
}  // namespace sb

using namespace sb;

extern "C" int sb_router_sizes(int64_t num_tokens, int32_t num_experts, int32_t k, int32_t tile, int32_t block_size,
                               int32_t ffn_dim, int64_t* max_assignments, int64_t* max_row_blocks, int64_t* max_rows,
                               int64_t* workspace_elems) {
  RouterSizes z;
  if (int rc = router_sizes(num_tokens, num_experts, k, tile, block_size, ffn_dim, &z)) return rc;
  if (max_assignments) *max_assignments = z.max_assignments;
  if (max_row_blocks) *max_row_blocks = z.max_row_blocks;
  if (max_rows) *max_rows = z.max_rows;
  if (workspace_elems) *workspace_elems = z.workspace_elems;
  return clear_ok();
}

extern "C" int sb_router_topk(const float* scores, int64_t num_tokens, int32_t num_experts, int32_t k,
                              int32_t* top_idx, float* top_weight, void* stream) {
  if (num_tokens <= 0 || num_tokens > 2147483647LL / 16) return fail(SB_ERR_INVALID, "scores must be [T, E] with T > 0");
  if (num_experts <= 0 || num_experts > kMaxExperts)
    return fail(SB_ERR_INVALID, "num_experts must be in [1, %d], got %d", kMaxExperts, num_experts);
  if (k <= 0 || k > num_experts || k > 16) return fail(SB_ERR_INVALID, "k must be in [1, min(E, 16)], got %d", k);
  if (!scores || !top_idx || !top_weight) return fail(SB_ERR_INVALID, "router top-k: null buffer");
  if (int rc = launch_topk(scores, num_tokens, num_experts, k, nullptr, nullptr, top_idx, top_weight,
                           as_stream(stream)))
    return rc;
  return clear_ok();
}

extern "C" int sb_token_rounding(const float* scores, int64_t num_tokens, int32_t num_experts, int32_t k,
                                 int32_t tile, int32_t block_size, int32_t ffn_dim, int32_t* workspace,
                                 int32_t* token_of_copy, int32_t* expert_of_copy, float* weight_of_copy,
                                 int32_t* num_assignments, int32_t* token_offsets, int32_t* tokens_per_expert,
                                 int32_t* padded_offsets, int32_t* row_token, int32_t* copy_row,
                                 int32_t* row_block_expert, int32_t* row_offsets, int32_t* col_indices,
                                 int32_t* error, void* stream_ptr) {
  RouterSizes z;
  if (int rc = router_sizes(num_tokens, num_experts, k, tile, block_size, ffn_dim, &z)) return rc;
  if (!scores || !workspace || !token_of_copy || !expert_of_copy || !weight_of_copy || !num_assignments ||
      !token_offsets || !tokens_per_expert || !padded_offsets || !row_token || !copy_row || !row_block_expert ||
      !row_offsets || !col_indices || !error)
    return fail(SB_ERR_INVALID, "token rounding: null buffer");
  const hipStream_t s = as_stream(stream_ptr);
  const int64_t t = num_tokens;
  const int32_t e = num_experts;
  // Workspace carve-up (int32 elements; the float arrays share the 4-byte slots).
  int32_t* chunk_counts = workspace;
  float* shifted = reinterpret_cast<float*>(chunk_counts + z.chunks * e);
  uint32_t* keep_mask = reinterpret_cast<uint32_t*>(shifted + t * e);
  int32_t* keep_prefix = reinterpret_cast<int32_t*>(keep_mask + z.words * e);

  if (int rc = launch_topk(scores, t, e, k, shifted, chunk_counts, nullptr, nullptr, s)) return rc;
  router_targets_kernel<<<1, 1024, 0, s>>>(chunk_counts, static_cast<int32_t>(z.chunks), e, t, tile, block_size,
                                           tokens_per_expert, padded_offsets, error);
  if (int rc = check_launch("token rounding targets")) return rc;
  router_select_kernel<<<e, kSelectThreads, 0, s>>>(shifted, t, tokens_per_expert, padded_offsets, keep_mask,
                                                    keep_prefix, row_token);
  if (int rc = check_launch("token rounding select")) return rc;
  const int32_t ffn_blocks = ffn_dim / block_size;
  const int64_t layout_items = std::max<int64_t>(z.max_row_blocks * ffn_blocks + 1, z.max_rows);
  const int64_t emit_groups = z.words + (layout_items + kEmitThreads - 1) / kEmitThreads;
  auto emit = [&](auto per) {
    router_emit_kernel<decltype(per)::value><<<static_cast<uint32_t>(emit_groups), kEmitThreads, 0, s>>>(
        scores, t, e, keep_mask, keep_prefix, tokens_per_expert, padded_offsets, z.max_assignments, block_size,
        ffn_blocks, static_cast<int32_t>(z.max_row_blocks), z.max_rows, token_offsets, num_assignments,
        token_of_copy, expert_of_copy, weight_of_copy, copy_row, row_token, row_block_expert, row_offsets,
        col_indices);
  };
  if (e <= 64) emit(std::integral_constant<int, 1>{});
  else if (e <= 128) emit(std::integral_constant<int, 2>{});
  else if (e <= 256) emit(std::integral_constant<int, 4>{});
  else emit(std::integral_constant<int, kMaxPerLane>{});
  if (int rc = check_launch("token rounding list")) return rc;
  return clear_ok();
}
