// The MoE layer on a routing given as assignments (the path of
// sparsebench/moe.py:59-91 in the reference, moe_forward_assigned): copy c
// sends token[c] to expert[c] with weight[c]; a token may have any number of
// copies, including none.
//
// Routing is the top-k routing with k = 1 and token ids read from the list
// (sb_routing_assigned). What changes is the combine: a token's copies are
// no longer the k consecutive entries t*k .. t*k+k-1, so the reference sums
// them with index_add_ (atomics, order not fixed). Here two steps replace it:
//
//   token_csr   token_offsets[T+1] and token_copies, the copies of each token
//               in ascending copy order. Each workgroup takes a run of tokens
//               and reads the whole list, so no workgroup waits for another;
//               lists of 524288 copies or more are taken in passes.
//   combine     out[t] = bf16( sum over t's copies, in copy order, of
//               fp32(y[copy_row[c]]) * fp32(weight[c]) ); 0 for no copies.
//
// Both are deterministic: the same list gives the same bits on every run.
// A token's copies are summed in list order, as the reference's index_add_
// does on the CPU, so a top-k list gives exactly the top-k combine's result.

#include "common.hpp"

namespace sb {
namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kCsrMaxTokens = 8192;  // of one workgroup
constexpr int kCsrMaxCopies = 8192;  // of one workgroup, ranked in LDS
constexpr int kCsrMaxList = 64;      // of one token, ranked in LDS

// Token of copy c, or -1 when it is not listed: routing did not place it
// (copy_row < 0: a bad expert or token id, or a token >= valid_tokens) or its
// token is out of range.
template <typename Tok>
__device__ __forceinline__ int32_t listed_token(const Tok* __restrict__ token, const int32_t* __restrict__ copy_row,
                                                int64_t c, int64_t n, int32_t num_tokens) {
  const int64_t at = min(c, n - 1);  // no branch: the caller's loads wait together
  const int32_t row = copy_row[at];
  const Tok t = token[at];
  const bool listed = (c < n) & (row >= 0) & (t >= 0) & (t < static_cast<Tok>(num_tokens));
  return listed ? static_cast<int32_t>(t) : -1;
}

// PER copies a lane, THREADS apart from `base` on, their loads in flight
// together: each copy's token (-1: not listed) and, for the check of the order,
// that of the copy before it (-1 before the first).
template <typename Tok, int THREADS, int PER>
struct CopyBatch {
  int32_t t[PER], prev[PER];
  __device__ __forceinline__ void load(const Tok* __restrict__ token, const int32_t* __restrict__ copy_row,
                                       int64_t base, int64_t n, int32_t num_tokens) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    Tok before[PER];  // the wave's
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int64_t first = base + u * THREADS + 64 * wave;
      before[u] = token[first > 0 ? min(first, n) - 1 : 0];
      t[u] = listed_token(token, copy_row, base + u * THREADS + threadIdx.x, n, num_tokens);
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      // A copy before it that is not listed breaks the order by itself.
      const int32_t own = base + u * THREADS + 64 * wave > 0 ? static_cast<int32_t>(before[u]) : -1;
      const int32_t below = __shfl_up(t[u], 1, 64);
      prev[u] = (threadIdx.x & 63) == 0 ? own : below;
    }
  }
};

// Workgroup g takes tokens g * per .. +per and reads the whole list, so the
// workgroups need nothing from each other. In a list already in token order
// (a top-k or a rounded list) the copies are 0, 1, 2, ... and each token starts
// where the token changes. Otherwise one pass counts the workgroup's tokens'
// copies in LDS and the listed copies of the tokens before them, which is where
// its copies start; a second pass gathers its copies into their tokens'
// slots, and each copy then moves to its rank within its token, so the order
// does not depend on timing. Bound by the latency of the list's loads (12 bytes
// a copy, from L2): a list of up to 8192 copies is held in registers (WHOLE),
// no more of them a lane than it needs (1024 copies in order 3.0 us with one a
// lane, 3.3 with 256 lanes of four, 4.7 with eight). 512 copies of 256 tokens
// in order 2.8 us, shuffled 5.6; 8192 of 4096 5.2 and 8.7 (one workgroup with
// global atomics 7.1 and 42); 65536 of 8192 23.4 and 34.9 (42 and 472).
// Lists longer than kCsrMaxList, where the ranks cost more than they save,
// and workgroups with more copies than the LDS holds take the slots in list
// order instead, wave after wave.
template <typename Tok, int THREADS, int PER, bool WHOLE>
__global__ void __launch_bounds__(THREADS)
    token_csr_kernel(const Tok* __restrict__ token, const int32_t* __restrict__ copy_row, int64_t n,
                     int32_t num_tokens, int32_t per, int32_t* __restrict__ offsets, int32_t* __restrict__ copies) {
  constexpr int kWaves = THREADS / 64;
  __shared__ int32_t start[kCsrMaxTokens + 1];  // counts, then first slots (the workgroup's own numbering)
  __shared__ int32_t next[kCsrMaxTokens];       // next free slot
  __shared__ int32_t buf[kCsrMaxCopies];
  __shared__ uint16_t buf_token[kCsrMaxCopies];
  __shared__ int32_t sums[3][kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t lo = static_cast<int32_t>(blockIdx.x) * per;
  const int32_t mine = min(per, num_tokens - lo);
  CopyBatch<Tok, THREADS, PER> batch;
  if constexpr (WHOLE) batch.load(token, copy_row, 0, n, num_tokens);
  // f(copy, its token, the token before it) for every copy.
  auto for_each_copy = [&](auto&& f) {
    for (int64_t base = 0; base < n; base += PER * THREADS) {
      if constexpr (!WHOLE) batch.load(token, copy_row, base, n, num_tokens);
#pragma unroll
      for (int u = 0; u < PER; ++u) f(static_cast<int32_t>(base + u * THREADS + tid), batch.t[u], batch.prev[u]);
      if constexpr (WHOLE) break;
    }
  };
  auto in_order = [&](int32_t c, int32_t t, int32_t prev) { return c >= n || (t >= 0 && t >= prev); };
  bool ordered = true;
  if constexpr (WHOLE) {
    const int32_t last = static_cast<int32_t>(token[n - 1]);  // a token of the list if it is in order
    for_each_copy([&](int32_t c, int32_t t, int32_t prev) { ordered = ordered && in_order(c, t, prev); });
    if (__syncthreads_and(ordered)) {
      for_each_copy([&](int32_t c, int32_t t, int32_t prev) {
        if (c >= n) return;
        if (t >= lo && t - lo < mine) copies[c] = c;
        for (int32_t u = max(prev + 1, lo); u <= min(t, lo + mine - 1); ++u) offsets[u] = c;
      });
      for (int32_t u = max(last + 1 - lo, 0) + tid; u < mine; u += THREADS) offsets[lo + u] = static_cast<int32_t>(n);
      if (lo + mine == num_tokens && tid == 0) offsets[num_tokens] = static_cast<int32_t>(n);
      return;
    }
  }

  for (int i = tid; i < mine; i += THREADS) start[i] = 0;
  __syncthreads();
  int32_t before = 0, all = 0;
  for_each_copy([&](int32_t c, int32_t t, int32_t prev) {
    all += t >= 0;
    before += t >= 0 && t < lo;
    if (t >= lo && t - lo < mine) atomicAdd(&start[t - lo], 1);
    ordered = ordered && in_order(c, t, prev);
  });
  for (int d = 32; d >= 1; d >>= 1) {
    before += __shfl_xor(before, d, 64);
    all += __shfl_xor(all, d, 64);
  }
  if (lane == 0) {
    sums[0][wave] = before;
    sums[1][wave] = all;
  }
  ordered = __syncthreads_and(ordered);
  before = all = 0;
  for (int w = 0; w < kWaves; ++w) {
    before += sums[0][w];
    all += sums[1][w];
  }

  // start[i] = slots before token lo + i.
  int32_t carry = 0;
  bool long_list = false;
  for (int32_t base = 0; base < mine; base += THREADS) {
    const int32_t i = base + tid;
    const int32_t own = i < mine ? start[i] : 0;
    long_list = long_list || own > kCsrMaxList;
    int32_t v = own;
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t below = __shfl_up(v, d, 64);
      if (lane >= d) v += below;
    }
    if (lane == 63) sums[2][wave] = v;
    __syncthreads();
    int32_t sum = 0;
    for (int w = 0; w < kWaves; ++w) {
      if (w < wave) v += sums[2][w];
      sum += sums[2][w];
    }
    if (i < mine) {
      start[i] = next[i] = carry + v - own;
      offsets[lo + i] = before + carry + v - own;
    }
    carry += sum;
    if (base + THREADS < mine) __syncthreads();  // sums[2] is written again
  }
  if (tid == 0) {
    start[mine] = carry;
    if (lo + mine == num_tokens) offsets[num_tokens] = all;
  }
  const bool by_list = __syncthreads_or(long_list || carry > kCsrMaxCopies);
  if (ordered) {  // every copy listed, in token order: a run of the list
    for (int32_t i = tid; i < carry; i += THREADS) copies[before + i] = before + i;
  } else if (!by_list) {
    for_each_copy([&](int32_t c, int32_t t, int32_t) {
      if (t >= lo && t - lo < mine) {
        const int32_t slot = atomicAdd(&next[t - lo], 1);
        buf[slot] = c;
        buf_token[slot] = static_cast<uint16_t>(t - lo);
      }
    });
    __syncthreads();
    for (int32_t i = tid; i < carry; i += THREADS) {
      const int32_t c = buf[i], s = start[buf_token[i]], e = start[buf_token[i] + 1];
      int32_t rank = 0;
      for (int32_t j = s; j < e; ++j) rank += buf[j] < c;
      copies[before + s + rank] = c;
    }
  } else {
    int bits = 0;
    while ((1 << bits) < mine) ++bits;
    for (int64_t base = 0; base < n; base += THREADS) {
      const int64_t c = base + tid;
      const int32_t t = listed_token(token, copy_row, c, n, num_tokens) - lo;
      const bool own = t >= 0 && t < mine;
      uint64_t peers = __ballot(own);  // the wave's lanes with a copy of the same token
      for (int b = 0; b < bits; ++b) {
        const uint64_t ones = __ballot(own && ((t >> b) & 1));
        peers &= ((t >> b) & 1) ? ones : ~ones;
      }
      const uint64_t lower = peers & ((uint64_t{1} << lane) - 1);
      for (int w = 0; w < kWaves; ++w) {
        if (w == wave && own) {
          const int32_t slot = next[t];
          copies[before + slot + __popcll(lower)] = static_cast<int32_t>(c);
          if (lower == 0) next[t] = slot + __popcll(peers);
        }
        __syncthreads();
      }
    }
  }
  // Unused tail of the copy list, shared by the workgroups.
  for (int64_t c = static_cast<int64_t>(all) + static_cast<int64_t>(blockIdx.x) * THREADS + tid; c < n;
       c += static_cast<int64_t>(gridDim.x) * THREADS)
    copies[c] = -1;
}

// Tokens of one workgroup: 128 while that is at most one workgroup a CU,
// then an equal share each, up to what its LDS holds, and fewer when they have
// so many copies that half of the LDS would not hold them.
int32_t csr_tokens_per_group(int64_t num_tokens, int64_t num_copies) {
  const int64_t share = std::min<int64_t>(std::max<int64_t>(128, (num_tokens + 255) / 256), kCsrMaxTokens);
  return static_cast<int32_t>(std::max<int64_t>(1, std::min(share, kCsrMaxCopies / 2 * num_tokens / num_copies)));
}

// Long lists, in passes over the list and the tokens whose work grows with
// their lengths alone (each workgroup reading the whole list makes it grow with
// the list's square: 8 million copies of a million tokens in order 18.1 ms,
// against 2.05 in passes, and 9.9 for one workgroup; 524288 of 65536 156 us
// against 173, shuffled 233 against 144, with one token of 65 copies 1010
// against 145):
// offsets as counts, scanned to the tokens' ends, which the placing of the
// copies walks down to their starts; then each token's copies into list order.
constexpr int64_t kCsrPassCopies = int64_t{1} << 19;
constexpr int kPassThreads = 1024;

__global__ void __launch_bounds__(kPassThreads) csr_clear_kernel(int32_t* __restrict__ offsets, int64_t count) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kPassThreads + threadIdx.x; i < count;
       i += static_cast<int64_t>(gridDim.x) * kPassThreads)
    offsets[i] = 0;
}

// PLACE false: offsets[t] counts token t's listed copies. PLACE true: each
// copy takes the slot below its token's end. One atomic a wave where all of
// it has the same token.
template <typename Tok, bool PLACE>
__global__ void __launch_bounds__(kPassThreads)
    csr_copies_kernel(const Tok* __restrict__ token, const int32_t* __restrict__ copy_row, int64_t n,
                      int32_t num_tokens, int32_t* __restrict__ offsets, int32_t* __restrict__ copies) {
  const int lane = threadIdx.x & 63;
  for (int64_t base = static_cast<int64_t>(blockIdx.x) * kPassThreads; base < n;
       base += static_cast<int64_t>(gridDim.x) * kPassThreads) {
    const int64_t c = base + threadIdx.x;
    const int32_t t = listed_token(token, copy_row, c, n, num_tokens);
    const int32_t one = __builtin_amdgcn_readfirstlane(t);
    if (one >= 0 && __ballot(t != one) == 0) {
      int32_t slot = 0;
      if (lane == 0) slot = PLACE ? atomicSub(&offsets[one], 64) - 64 : atomicAdd(&offsets[one], 64);
      if (PLACE) copies[__builtin_amdgcn_readfirstlane(slot) + lane] = static_cast<int32_t>(c);
    } else if (t >= 0) {
      if (PLACE) copies[atomicSub(&offsets[t], 1) - 1] = static_cast<int32_t>(c);
      else atomicAdd(&offsets[t], 1);
    }
  }
}

// Inclusive scan of offsets[0 .. num_tokens] in place, by one workgroup.
__global__ void __launch_bounds__(kPassThreads) csr_scan_kernel(int32_t* __restrict__ offsets, int64_t count) {
  constexpr int kPer = 16;
  __shared__ int32_t wave_sums[2][kPassThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int32_t carry = 0;
  int turn = 0;
  for (int64_t base = 0; base < count; base += kPer * kPassThreads, turn ^= 1) {
    const int64_t first = base + static_cast<int64_t>(tid) * kPer;
    int32_t v[kPer], own = 0;
#pragma unroll
    for (int u = 0; u < kPer; ++u) v[u] = first + u < count ? offsets[first + u] : 0;
#pragma unroll
    for (int u = 0; u < kPer; ++u) own += v[u];
    int32_t incl = own;
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t below = __shfl_up(incl, d, 64);
      if (lane >= d) incl += below;
    }
    if (lane == 63) wave_sums[turn][wave] = incl;
    __syncthreads();  // the other turn's sums have been read by all before this
    int32_t run = carry + incl - own;
    for (int w = 0; w < kPassThreads / 64; ++w) {
      if (w < wave) run += wave_sums[turn][w];
      carry += wave_sums[turn][w];
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      run += v[u];
      if (first + u < count) offsets[first + u] = run;
    }
  }
}

// Each token's copies into ascending order, a lane a token; longer lists than
// kCsrMaxList are left to csr_order_long_kernel. The tail past the listed copies
// gets -1.
__global__ void __launch_bounds__(kPassThreads)
    csr_order_kernel(int64_t n, int32_t num_tokens, const int32_t* __restrict__ offsets, int32_t* __restrict__ copies) {
  const int64_t own = static_cast<int64_t>(blockIdx.x) * kPassThreads + threadIdx.x;
  if (own < num_tokens) {
    const int32_t s = offsets[own], e = offsets[own + 1];
    if (e - s <= kCsrMaxList) {
      for (int32_t i = s + 1; i < e; ++i) {
        const int32_t v = copies[i];
        int32_t j = i - 1;
        for (; j >= s; --j) {
          const int32_t u = copies[j];
          if (u < v) break;
          copies[j + 1] = u;
        }
        copies[j + 1] = v;
      }
    }
  }
  const int64_t all = offsets[num_tokens];
  for (int64_t c = all + own; c < n; c += static_cast<int64_t>(gridDim.x) * kPassThreads) copies[c] = -1;
}

// The longer lists, each by a whole workgroup: in LDS or, past what it holds,
// from the list itself. A workgroup's tokens are gridDim.x apart, so that long
// lists side by side go to different ones.
template <typename Tok>
__global__ void __launch_bounds__(kPassThreads)
    csr_order_long_kernel(const Tok* __restrict__ token, const int32_t* __restrict__ copy_row, int64_t n,
                          int32_t num_tokens, const int32_t* __restrict__ offsets, int32_t* __restrict__ copies) {
  constexpr int kPer = 8;  // loads in flight
  constexpr int kWaves = kPassThreads / 64;
  __shared__ int32_t buf[kCsrMaxCopies];
  __shared__ int32_t long_tokens[kPassThreads];
  __shared__ int32_t num_long;
  __shared__ int32_t wave_counts[kPer * kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t stride = gridDim.x;
  for (int64_t base = blockIdx.x; base < num_tokens; base += stride * kPassThreads) {
    if (tid == 0) num_long = 0;
    __syncthreads();
    const int64_t own = base + stride * tid;
    if (own < num_tokens && offsets[own + 1] - offsets[own] > kCsrMaxList)
      long_tokens[atomicAdd(&num_long, 1)] = static_cast<int32_t>(own);
    __syncthreads();
    const int count = num_long;
    for (int i = 0; i < count; ++i) {
      const int32_t t = long_tokens[i], s = offsets[t], len = offsets[t + 1] - s;
      if (len <= kCsrMaxCopies) {  // bitonic sort, padded with the largest value
        int size = 2 * kCsrMaxList;
        while (size < len) size *= 2;
        for (int j = tid; j < size; j += kPassThreads) buf[j] = j < len ? copies[s + j] : 0x7fffffff;
        __syncthreads();
        for (int k = 2; k <= size; k *= 2)
          for (int d = k / 2; d >= 1; d /= 2) {
            for (int j = tid; j < size; j += kPassThreads) {
              const int other = j ^ d;
              const int32_t a = buf[j], b = buf[other];
              if (other > j && (a > b) == ((j & k) == 0)) {
                buf[j] = b;
                buf[other] = a;
              }
            }
            __syncthreads();
          }
        for (int j = tid; j < len; j += kPassThreads) copies[s + j] = buf[j];
      } else {
        int32_t slot = s;
        for (int64_t at = 0; at < n; at += kPer * kPassThreads) {
          uint64_t mine[kPer];
#pragma unroll
          for (int u = 0; u < kPer; ++u)
            mine[u] = __ballot(listed_token(token, copy_row, at + u * kPassThreads + tid, n, num_tokens) == t);
#pragma unroll
          for (int u = 0; u < kPer; ++u)
            if (lane == 0) wave_counts[u * kWaves + wave] = __popcll(mine[u]);
          __syncthreads();
#pragma unroll
          for (int u = 0; u < kPer; ++u) {
            int32_t before = slot;
            for (int w = 0; w < kWaves; ++w) {
              const int32_t of_wave = wave_counts[u * kWaves + w];
              if (w < wave) before += of_wave;
              slot += of_wave;
            }
            if ((mine[u] >> lane) & 1)
              copies[before + __popcll(mine[u] & ((uint64_t{1} << lane) - 1))] =
                  static_cast<int32_t>(at + u * kPassThreads + tid);
          }
          __syncthreads();
        }
      }
      __syncthreads();
    }
  }
}

template <typename Tok>
int launch_token_csr(const Tok* token, const int32_t* copy_row, int64_t n, int64_t num_tokens, int32_t* offsets,
                     int32_t* copies, hipStream_t s) {
  const int32_t tokens = static_cast<int32_t>(num_tokens);
  if (n < kCsrPassCopies) {
    const int32_t per = csr_tokens_per_group(num_tokens, n);
    const uint32_t groups = static_cast<uint32_t>((num_tokens + per - 1) / per);
    auto launch = [&](auto threads, auto copies_a_lane, auto whole) {
      constexpr int kThreads = decltype(threads)::value;
      token_csr_kernel<Tok, kThreads, decltype(copies_a_lane)::value, decltype(whole)::value>
          <<<groups, kThreads, 0, s>>>(token, copy_row, n, tokens, per, offsets, copies);
    };
    const std::integral_constant<int, 1024> wide;
    if (n <= 256) launch(std::integral_constant<int, 256>{}, std::integral_constant<int, 1>{}, std::true_type{});
    else if (n <= 1024) launch(wide, std::integral_constant<int, 1>{}, std::true_type{});
    else if (n <= 2048) launch(wide, std::integral_constant<int, 2>{}, std::true_type{});
    else if (n <= 4096) launch(wide, std::integral_constant<int, 4>{}, std::true_type{});
    else if (n <= 8192) launch(wide, std::integral_constant<int, 8>{}, std::true_type{});
    else launch(wide, std::integral_constant<int, 8>{}, std::false_type{});
    return check_launch("token_csr");
  }
  auto groups = [](int64_t items, int64_t most) {
    return static_cast<uint32_t>(std::min((items + kPassThreads - 1) / kPassThreads, most));
  };
  constexpr int64_t kPassGroups = 2048;  // of grid-strided passes
  csr_clear_kernel<<<groups(num_tokens + 1, kPassGroups), kPassThreads, 0, s>>>(offsets, num_tokens + 1);
  if (int rc = check_launch("token_csr clear")) return rc;
  csr_copies_kernel<Tok, false><<<groups(n, kPassGroups), kPassThreads, 0, s>>>(token, copy_row, n, tokens, offsets,
                                                                                copies);
  if (int rc = check_launch("token_csr count")) return rc;
  csr_scan_kernel<<<1, kPassThreads, 0, s>>>(offsets, num_tokens + 1);
  if (int rc = check_launch("token_csr scan")) return rc;
  csr_copies_kernel<Tok, true><<<groups(n, kPassGroups), kPassThreads, 0, s>>>(token, copy_row, n, tokens, offsets,
                                                                               copies);
  if (int rc = check_launch("token_csr place")) return rc;
  csr_order_kernel<<<groups(num_tokens, int64_t{1} << 31), kPassThreads, 0, s>>>(n, tokens, offsets, copies);
  if (int rc = check_launch("token_csr order")) return rc;
  csr_order_long_kernel<Tok><<<static_cast<uint32_t>(std::min(num_tokens, kPassGroups)), kPassThreads, 0, s>>>(
      token, copy_row, n, tokens, offsets, copies);
  return check_launch("token_csr order of long lists");
}

template <typename G>
__device__ __forceinline__ float weight_f32(const G* g, int64_t i);
template <>
__device__ __forceinline__ float weight_f32<uint16_t>(const uint16_t* g, int64_t i) {
  return bf16_to_f32(g[i]);
}
template <>
__device__ __forceinline__ float weight_f32<_Float16>(const _Float16* g, int64_t i) {
  return static_cast<float>(g[i]);
}
template <>
__device__ __forceinline__ float weight_f32<float>(const float* g, int64_t i) {
  return g[i];
}

// One lane per 16 bytes (8 columns) of one token row.
template <typename G>
__global__ void __launch_bounds__(256)
    combine_assigned_kernel(const uint16_t* __restrict__ y, const int32_t* __restrict__ copy_row,
                            const G* __restrict__ weights, const int32_t* __restrict__ offsets,
                            const int32_t* __restrict__ copies, uint16_t* __restrict__ out, int64_t num_tokens,
                            int32_t chunks_per_row, int64_t y_rows, const int32_t* __restrict__ valid_tokens) {
  // Products rounded, then added (no fused multiply-add), as the reference's
  // index_add_ of rows.float() * weight.
#pragma clang fp contract(off)
  const int64_t item = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t t = item / chunks_per_row;
  const int32_t ch = static_cast<int32_t>(item % chunks_per_row);
  const int64_t limit = valid_tokens ? min(num_tokens, static_cast<int64_t>(*valid_tokens)) : num_tokens;
  if (t >= limit) return;
  const int64_t d_model = static_cast<int64_t>(chunks_per_row) * 8;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const int32_t s = offsets[t], e = offsets[t + 1];
  for (int32_t i = s; i < e; ++i) {
    const int32_t c = copies != nullptr ? copies[i] : i;  // no list: copies already in token order
    const int32_t row = c >= 0 ? copy_row[c] : -1;
    if (row < 0 || row >= y_rows) continue;
    const float g = weight_f32(weights, c);
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(y + row * d_model + ch * 8);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      acc[2 * q] += __uint_as_float(v[q] << 16) * g;
      acc[2 * q + 1] += __uint_as_float(v[q] & 0xffff0000u) * g;
    }
  }
  u32x4_t o;
#pragma unroll
  for (int q = 0; q < 4; ++q) o[q] = pack_bf16x2(acc[2 * q], acc[2 * q + 1]);
  *reinterpret_cast<u32x4_t*>(out + t * d_model + ch * 8) = o;
}

template <typename G>
int launch_combine_assigned(const void* y, const int32_t* copy_row, const void* weights, const int32_t* offsets,
                            const int32_t* copies, void* out, int64_t num_tokens, int64_t d_model, int64_t y_rows,
                            const int32_t* valid_tokens, hipStream_t stream) {
  const int32_t chunks = static_cast<int32_t>(d_model / 8);
  const int64_t groups = (num_tokens * chunks + 255) / 256;
  combine_assigned_kernel<G><<<static_cast<uint32_t>(groups), 256, 0, stream>>>(
      static_cast<const uint16_t*>(y), copy_row, static_cast<const G*>(weights), offsets, copies,
      static_cast<uint16_t*>(out), num_tokens, chunks, y_rows, valid_tokens);
  return check_launch("combine (assigned)");
}

}  // namespace
}  // namespace sb

using namespace sb;

extern "C" int sb_token_csr(const void* token_of_copy, int32_t token_is_i64, const int32_t* copy_row,
                            int64_t num_copies, int64_t num_tokens, int32_t* token_offsets, int32_t* token_copies,
                            void* stream) {
  if (num_copies <= 0 || num_copies > 2147483647LL) return fail(SB_ERR_INVALID, "token_csr: bad copy count");
  if (num_tokens <= 0 || num_tokens > 2147483646LL) return fail(SB_ERR_INVALID, "token_csr: bad token count");
  if (!token_of_copy || !copy_row || !token_offsets || !token_copies)
    return fail(SB_ERR_INVALID, "token_csr: null buffer");
  const hipStream_t s = as_stream(stream);
  const int rc = token_is_i64 ? launch_token_csr(static_cast<const int64_t*>(token_of_copy), copy_row, num_copies,
                                                 num_tokens, token_offsets, token_copies, s)
                              : launch_token_csr(static_cast<const int32_t*>(token_of_copy), copy_row, num_copies,
                                                 num_tokens, token_offsets, token_copies, s);
  return rc ? rc : clear_ok();
}

extern "C" int sb_combine_assigned(const void* y, const int32_t* copy_row, const void* weights, int32_t weight_dtype,
                                   const int32_t* token_offsets, const int32_t* token_copies, void* out,
                                   int64_t num_tokens, int64_t d_model, int64_t y_rows, const int32_t* valid_tokens,
                                   void* stream) {
  if (num_tokens < 0) return fail(SB_ERR_INVALID, "combine: bad token count");
  if (d_model <= 0 || d_model % 8 != 0)
    return fail(SB_ERR_INVALID, "combine: D (%lld) must be a positive multiple of 8", static_cast<long long>(d_model));
  if (num_tokens == 0) return clear_ok();
  if (!y || !copy_row || !weights || !token_offsets || !out) return fail(SB_ERR_INVALID, "combine: null buffer");
  if (!aligned16(y) || !aligned16(out)) return fail(SB_ERR_INVALID, "combine: y and out must be 16-byte aligned");
  if ((num_tokens * (d_model / 8) + 255) / 256 > 2147483647LL) return fail(SB_ERR_INVALID, "combine: too many tokens");
  const hipStream_t s = as_stream(stream);
  switch (weight_dtype) {
    case SB_DTYPE_BF16:
      return launch_combine_assigned<uint16_t>(y, copy_row, weights, token_offsets, token_copies, out, num_tokens,
                                               d_model, y_rows, valid_tokens, s);
    case SB_DTYPE_F16:
      return launch_combine_assigned<_Float16>(y, copy_row, weights, token_offsets, token_copies, out, num_tokens,
                                               d_model, y_rows, valid_tokens, s);
    case SB_DTYPE_F32:
      return launch_combine_assigned<float>(y, copy_row, weights, token_offsets, token_copies, out, num_tokens,
                                            d_model, y_rows, valid_tokens, s);
    default:
      return fail(SB_ERR_INVALID, "combine: unsupported weight dtype code %d", weight_dtype);
  }
}
