// One SDD / DSD tile of a chunk of an expert's rows on the LDS-DMA main loop
// (gemm_dma.hpp), for any tile configuration: the layer kernels' expert
// chunks, row blocks and narrow tiles (experts.hip).
#pragma once

#include "expert_chunks.hpp"
#include "gelu.hpp"
#include "gemm_dma.hpp"

namespace sb {

// A tile configuration cut to R row groups (R a multiple of its rows of
// waves, WM: DmaCfg asserts that each wave owns whole 32-row groups).
template <class Cfg, int R>
using RowsCfg = DmaCfg<32 * R, Cfg::BN, Cfg::BK, Cfg::STAGES, Cfg::WM, Cfg::WN, Cfg::CPA, Cfg::CPB, Cfg::PIPE,
                       Cfg::EPI_PARTS, Cfg::APAIR ? 1 : 0, Cfg::BSTAGES == Cfg::STAGES ? 0 : Cfg::BSTAGES>;

// f(integral_constant<int, R>) for the chunk's R in 1 .. RMAX.
template <int RMAX, class F>
__device__ __forceinline__ void with_groups(int groups, F&& f) {
  static_for<1, RMAX + 1>([&](auto rc) {
    constexpr int R = decltype(rc)::value;
    if (groups == R) f(rc);
  });
}

// ------------------------------------------------------------------ SDD ---

template <class Cfg>
struct SddChunkSrc {
  __amdgpu_buffer_rsrc_t x_rsrc, w_rsrc;
  uint32_t a_off[Cfg::kAInstr];
  uint32_t b_off[Cfg::kBInstr];
  uint32_t b_step_bytes;
  __device__ __forceinline__ uint32_t a_voff(int q) const { return a_off[q]; }
  __device__ __forceinline__ uint32_t b_voff(int q) const { return b_off[q]; }
  __device__ __forceinline__ void a_src(int t, __amdgpu_buffer_rsrc_t* r, uint32_t* s) const {
    *r = x_rsrc;
    *s = static_cast<uint32_t>(t) * (Cfg::BK * 2);
  }
  __device__ __forceinline__ void b_src(int t, __amdgpu_buffer_rsrc_t* r, uint32_t* s) const {
    *r = w_rsrc;
    *s = static_cast<uint32_t>(t) * b_step_bytes;
  }
};

struct SddArgs {
  const uint16_t* x;
  const uint16_t* w1;
  const int32_t* row_token;
  uint16_t* out;
  int32_t num_tokens, d_model, ffn_dim;
  int32_t apply_gelu;
};

template <class Cfg>
__device__ __forceinline__ void sdd_chunk_tile(uint8_t* __restrict__ lds, const SddArgs& a, const Chunk& ch, int n0) {
  using ML = DmaMainloop<Cfg>;
  SddChunkSrc<Cfg> src;
  src.x_rsrc = make_rsrc(a.x, static_cast<uint32_t>(a.num_tokens) * static_cast<uint32_t>(a.d_model) * 2u);
  src.w_rsrc = make_rsrc(a.w1 + static_cast<int64_t>(ch.expert) * a.d_model * a.ffn_dim,
                         static_cast<uint32_t>(a.d_model) * static_cast<uint32_t>(a.ffn_dim) * 2u);
  src.b_step_bytes = static_cast<uint32_t>(Cfg::BK) * static_cast<uint32_t>(a.ffn_dim) * 2u;
  const ADmaPos<Cfg> ap;
#pragma unroll
  for (int q = 0; q < Cfg::kAInstr; ++q) {
    const int j = ap.row[q];  // row of the chunk; rows past BM belong to the rounded-up DMA area
    const int32_t tok = j < ch.rows ? a.row_token[ch.row0 + j] : -1;
    src.a_off[q] = (tok >= 0 && tok < a.num_tokens)
                       ? static_cast<uint32_t>(tok) * static_cast<uint32_t>(a.d_model) * 2u + ap.chunk[q] * 16u
                       : kOutOfRange;
  }
  const BDmaPos<Cfg> bp;
#pragma unroll
  for (int q = 0; q < Cfg::kBInstr; ++q)
    src.b_off[q] = (static_cast<uint32_t>(bp.row[q]) * a.ffn_dim + n0 + bp.col[q]) * 2u;

  typename ML::Acc acc;
  ML::run(lds, src, a.d_model / Cfg::BK, acc);

  // Padded row p -> row block p / 128, whose blocks are (p / 128) * F/128 + f/128.
  const int64_t ffn_blocks = a.ffn_dim / kBS;
  static_for<0, Cfg::EPI_PARTS>([&](auto pc) {
    constexpr int P = decltype(pc)::value;
    if (a.apply_gelu)
      ML::template stage_part<P>(lds, acc, [](float v) { return gelu_erf_fast(v); });
    else
      ML::template stage_part<P>(lds, acc, [](float v) { return v; });
    ML::for_each_staged_chunk(lds, [&](int m, int col, u32x4_t v) {
      const int p = ch.row0 + P * ML::kPartRows + m;
      const int f = n0 + col;
      *reinterpret_cast<u32x4_t*>(a.out + ((p / kBS) * ffn_blocks + f / kBS) * (kBS * kBS) + (p % kBS) * kBS +
                                  (f % kBS)) = v;
    });
  });
}

// ------------------------------------------------------------------ DSD ---

// A: the chunk's rows of H, read in place. All of H is one buffer; lane row
// j of the chunk sits in row block row0/128 + j/128 at row j % 128, so its
// offset from the chunk's first block of the K step is fixed per lane, and
// the step moves the scalar offset (4 steps of 32 per 128-wide block).
template <class Cfg>
struct DsdChunkSrc {
  static constexpr int kStepsPerBlock = kBS / Cfg::BK;
  __amdgpu_buffer_rsrc_t h_rsrc, w_rsrc;
  uint32_t h_base;  // byte offset of the chunk's first H block
  uint32_t w_step_bytes, n0_bytes;
  uint32_t a_off[Cfg::kAInstr];
  uint32_t b_off[Cfg::kBInstr];
  __device__ __forceinline__ uint32_t a_voff(int q) const { return a_off[q]; }
  __device__ __forceinline__ uint32_t b_voff(int q) const { return b_off[q]; }
  __device__ __forceinline__ void a_src(int t, __amdgpu_buffer_rsrc_t* r, uint32_t* s) const {
    *r = h_rsrc;
    *s = h_base + static_cast<uint32_t>(t / kStepsPerBlock) * (kBS * kBS * 2) +
         static_cast<uint32_t>(t % kStepsPerBlock) * (Cfg::BK * 2);
  }
  __device__ __forceinline__ void b_src(int t, __amdgpu_buffer_rsrc_t* r, uint32_t* s) const {
    *r = w_rsrc;
    *s = static_cast<uint32_t>(t) * w_step_bytes + n0_bytes;
  }
};

struct DsdArgs {
  const uint16_t* h;
  const uint16_t* w2;
  uint16_t* out;
  int64_t h_bytes;
  int32_t ffn_dim, d_model;
};

template <class Cfg>
__device__ __forceinline__ void dsd_chunk_tile(uint8_t* __restrict__ lds, const DsdArgs& a, const Chunk& ch, int n0) {
  using ML = DmaMainloop<Cfg>;
  const uint32_t ffn_blocks = static_cast<uint32_t>(a.ffn_dim / kBS);
  DsdChunkSrc<Cfg> src;
  src.h_rsrc = make_rsrc(a.h, static_cast<uint32_t>(a.h_bytes));
  src.h_base = static_cast<uint32_t>(ch.row0 / kBS) * ffn_blocks * (kBS * kBS * 2);
  src.w_rsrc = make_rsrc(a.w2 + static_cast<int64_t>(ch.expert) * a.ffn_dim * a.d_model,
                         static_cast<uint32_t>(a.ffn_dim) * static_cast<uint32_t>(a.d_model) * 2u);
  src.w_step_bytes = static_cast<uint32_t>(Cfg::BK) * static_cast<uint32_t>(a.d_model) * 2u;
  src.n0_bytes = static_cast<uint32_t>(n0) * 2u;
  const ADmaPos<Cfg> ap;
#pragma unroll
  for (int q = 0; q < Cfg::kAInstr; ++q) {
    const uint32_t j = static_cast<uint32_t>(ap.row[q]);
    src.a_off[q] = static_cast<int>(j) < ch.rows
                       ? ((j / kBS) * ffn_blocks * (kBS * kBS) + (j % kBS) * kBS) * 2u + ap.chunk[q] * 16u
                       : kOutOfRange;
  }
  const BDmaPos<Cfg> bp;
#pragma unroll
  for (int q = 0; q < Cfg::kBInstr; ++q)
    src.b_off[q] = (static_cast<uint32_t>(bp.row[q]) * a.d_model + bp.col[q]) * 2u;

  typename ML::Acc acc;
  ML::run(lds, src, a.ffn_dim / Cfg::BK, acc);

  ML::stage_tile(lds, acc, [](float v) { return v; });
  uint16_t* out_tile = a.out + static_cast<int64_t>(ch.row0) * a.d_model + n0;
  ML::for_each_staged_chunk(lds, [&](int m, int col, u32x4_t v) {
    if (m < ch.rows) *reinterpret_cast<u32x4_t*>(out_tile + static_cast<int64_t>(m) * a.d_model + col) = v;
  });
}

}  // namespace sb
