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
//               and reads the whole list, so no workgroup waits for another.
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

constexpr int kCsrThreads = 1024;
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

// f(c, token) for every copy, lane-strided, kPer copies' loads in flight at
// once (token -1: not listed).
template <typename Tok, class F>
__device__ __forceinline__ void for_each_copy(const Tok* __restrict__ token, const int32_t* __restrict__ copy_row,
                                              int64_t n, int32_t num_tokens, F&& f) {
  constexpr int kPer = 8;
  for (int64_t base = threadIdx.x; base < n; base += kPer * kCsrThreads) {
    int32_t t[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) t[u] = listed_token(token, copy_row, base + u * kCsrThreads, n, num_tokens);
#pragma unroll
    for (int u = 0; u < kPer; ++u) f(static_cast<int32_t>(base + u * kCsrThreads), t[u]);
  }
}

// Sum of v over the workgroup, in every lane.
__device__ __forceinline__ int32_t block_sum(int32_t v, int32_t* wave_sums) {
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  if ((threadIdx.x & 63) == 0) wave_sums[threadIdx.x >> 6] = v;
  __syncthreads();
  int32_t sum = 0;
  for (int w = 0; w < kCsrThreads / 64; ++w) sum += wave_sums[w];
  __syncthreads();
  return sum;
}

// Workgroup g takes tokens g * per .. +per. One pass over the whole list
// counts its tokens' copies in LDS and the listed copies of the tokens
// before them, which is where its copies start, so the workgroups need
// nothing from each other; a second pass gathers its copies into their
// tokens' slots, and each copy then moves to its rank within its token, so
// the order does not depend on timing. (One workgroup with global atomics
// took 41.7 us for 8192 copies of 4096 tokens, bound by their latency; this
// takes 9.8: the list is read by every workgroup, 12 bytes a copy from L2.)
// In a list already in token order (a top-k or a rounded list) the copies
// are those slots themselves, and the second pass is left out.
// Lists longer than kCsrMaxList, where the ranks cost more than they save,
// and workgroups with more copies than the LDS holds take the slots in list
// order instead, wave after wave.
template <typename Tok>
__global__ void __launch_bounds__(kCsrThreads)
    token_csr_kernel(const Tok* __restrict__ token, const int32_t* __restrict__ copy_row, int64_t n,
                     int32_t num_tokens, int32_t per, int32_t* __restrict__ offsets, int32_t* __restrict__ copies) {
  __shared__ int32_t start[kCsrMaxTokens + 1];  // counts, then first slots (the workgroup's own numbering)
  __shared__ int32_t next[kCsrMaxTokens];       // next free slot
  __shared__ int32_t buf[kCsrMaxCopies];
  __shared__ uint16_t buf_token[kCsrMaxCopies];
  __shared__ int32_t wave_sums[kCsrThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t lo = static_cast<int32_t>(blockIdx.x) * per;
  const int32_t mine = min(per, num_tokens - lo);
  for (int i = tid; i < mine; i += kCsrThreads) start[i] = 0;
  __syncthreads();

  int32_t before = 0, all = 0;
  bool ordered = true;
  for_each_copy(token, copy_row, n, num_tokens, [&](int32_t c, int32_t t) {
    all += t >= 0;
    before += t >= 0 && t < lo;
    if (t >= lo && t - lo < mine) atomicAdd(&start[t - lo], 1);
    // The token before it, from the lane below; a wave's first lane reads it.
    int32_t prev = __shfl_up(t, 1, 64);
    if (lane == 0) prev = c > 0 && c < n ? static_cast<int32_t>(token[c - 1]) : 0;
    ordered = ordered && (c >= n || (t >= 0 && t >= prev));
  });
  before = block_sum(before, wave_sums);  // synchronizes the workgroup
  all = block_sum(all, wave_sums);

  // start[i] = slots before token lo + i.
  int32_t carry = 0;
  bool long_list = false;
  for (int32_t base = 0; base < mine; base += kCsrThreads) {
    const int32_t i = base + tid;
    const int32_t own = i < mine ? start[i] : 0;
    long_list = long_list || own > kCsrMaxList;
    int32_t v = own;
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t below = __shfl_up(v, d, 64);
      if (lane >= d) v += below;
    }
    if (lane == 63) wave_sums[wave] = v;
    __syncthreads();
    int32_t sum = 0;
    for (int w = 0; w < kCsrThreads / 64; ++w) {
      if (w < wave) v += wave_sums[w];
      sum += wave_sums[w];
    }
    if (i < mine) {
      start[i] = next[i] = carry + v - own;
      offsets[lo + i] = before + carry + v - own;
    }
    carry += sum;
    __syncthreads();
  }
  if (tid == 0) {
    start[mine] = carry;
    if (lo + mine == num_tokens) offsets[num_tokens] = all;
  }
  if (__syncthreads_and(ordered)) {  // every copy listed, in token order: a run of the list
    for (int32_t i = tid; i < carry; i += kCsrThreads) copies[before + i] = before + i;
  } else if (!__syncthreads_or(long_list || carry > kCsrMaxCopies)) {
    for_each_copy(token, copy_row, n, num_tokens, [&](int32_t c, int32_t t) {
      if (t >= lo && t - lo < mine) {
        const int32_t slot = atomicAdd(&next[t - lo], 1);
        buf[slot] = c;
        buf_token[slot] = static_cast<uint16_t>(t - lo);
      }
    });
    __syncthreads();
    for (int32_t i = tid; i < carry; i += kCsrThreads) {
      const int32_t c = buf[i], s = start[buf_token[i]], e = start[buf_token[i] + 1];
      int32_t rank = 0;
      for (int32_t j = s; j < e; ++j) rank += buf[j] < c;
      copies[before + s + rank] = c;
    }
  } else {
    int bits = 0;
    while ((1 << bits) < mine) ++bits;
    for (int64_t base = 0; base < n; base += kCsrThreads) {
      const int64_t c = base + tid;
      const int32_t t = listed_token(token, copy_row, c, n, num_tokens) - lo;
      const bool own = t >= 0 && t < mine;
      uint64_t peers = __ballot(own);  // the wave's lanes with a copy of the same token
      for (int b = 0; b < bits; ++b) {
        const uint64_t ones = __ballot(own && ((t >> b) & 1));
        peers &= ((t >> b) & 1) ? ones : ~ones;
      }
      const uint64_t lower = peers & ((uint64_t{1} << lane) - 1);
      for (int w = 0; w < kCsrThreads / 64; ++w) {
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
  for (int64_t c = static_cast<int64_t>(all) + static_cast<int64_t>(blockIdx.x) * kCsrThreads + tid; c < n;
       c += static_cast<int64_t>(gridDim.x) * kCsrThreads)
    copies[c] = -1;
}

// Tokens of one workgroup: 128 while that is at most one workgroup a CU,
// then an equal share each, up to what its LDS holds, and fewer when they have
// so many copies that half of the LDS would not hold them.
int32_t csr_tokens_per_group(int64_t num_tokens, int64_t num_copies) {
  const int64_t share = std::min<int64_t>(std::max<int64_t>(128, (num_tokens + 255) / 256), kCsrMaxTokens);
  return static_cast<int32_t>(std::max<int64_t>(1, std::min(share, kCsrMaxCopies / 2 * num_tokens / num_copies)));
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
  const int32_t per = csr_tokens_per_group(num_tokens, num_copies);
  const uint32_t groups = static_cast<uint32_t>((num_tokens + per - 1) / per);
  if (token_is_i64)
    token_csr_kernel<int64_t><<<groups, kCsrThreads, 0, s>>>(static_cast<const int64_t*>(token_of_copy), copy_row,
                                                             num_copies, static_cast<int32_t>(num_tokens), per,
                                                             token_offsets, token_copies);
  else
    token_csr_kernel<int32_t><<<groups, kCsrThreads, 0, s>>>(static_cast<const int32_t*>(token_of_copy), copy_row,
                                                             num_copies, static_cast<int32_t>(num_tokens), per,
                                                             token_offsets, token_copies);
  if (int rc = check_launch("token_csr")) return rc;
  return clear_ok();
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
