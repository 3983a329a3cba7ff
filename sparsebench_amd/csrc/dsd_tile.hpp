// One DSD tile of a row block on the LDS-DMA main loop (gemm_dma.hpp), the
// tile of the per-row-block kernels (dsd.hip).
#pragma once

#include "gemm_dma.hpp"

namespace sb {

// The same tile on the LDS-DMA mainloop (gemm_dma.hpp). A block of w that
// does not exist (bad column index) gets a zero-length buffer: its loads
// return zeros and it contributes nothing.
template <class Cfg>
struct DsdDmaSrc {
  static constexpr int kStepsPerBlock = Cfg::BM / Cfg::BK;
  // A row block's reduction is whole blocks (reduction_fits for any count).
  static_assert(!Cfg::APAIR || kStepsPerBlock % 2 == 0, "paired A needs an even step count per block");
  const uint16_t* blocks;
  const uint16_t* w;
  const int32_t* col_indices;
  int64_t w_rows;
  int32_t d_model, begin;
  uint32_t a_off[Cfg::kAInstr];
  uint32_t b_off[Cfg::kBInstr];
  __device__ __forceinline__ uint32_t a_voff(int q) const { return a_off[q]; }
  __device__ __forceinline__ uint32_t b_voff(int q) const { return b_off[q]; }
  __device__ __forceinline__ void a_src(int t, __amdgpu_buffer_rsrc_t* r, uint32_t* s) const {
    const int32_t p = begin + t / kStepsPerBlock;
    *r = make_rsrc(blocks + static_cast<int64_t>(p) * Cfg::BM * Cfg::BM, Cfg::BM * Cfg::BM * 2);
    *s = static_cast<uint32_t>(t % kStepsPerBlock) * (Cfg::BK * 2);
  }
  __device__ __forceinline__ void b_src(int t, __amdgpu_buffer_rsrc_t* r, uint32_t* s) const {
    const int32_t p = begin + t / kStepsPerBlock;
    const int64_t row0 = static_cast<int64_t>(col_indices[p]) * Cfg::BM;
    const bool ok = row0 >= 0 && row0 + Cfg::BM <= w_rows;
    *r = make_rsrc(w + (ok ? row0 : 0) * d_model, ok ? static_cast<uint32_t>(Cfg::BM) * d_model * 2u : 0u);
    *s = static_cast<uint32_t>(t % kStepsPerBlock) * (Cfg::BK * 2u) * static_cast<uint32_t>(d_model);
  }
};

// Tile `tile_id` of the row-block grid: bs x BN outputs of one row block,
// its blocks walked in K steps through col_indices. Ids past the grid's
// num_row_blocks * num_slices tiles do nothing.
template <class Cfg>
__device__ __forceinline__ void dsd_row_block_tile(uint8_t* __restrict__ lds, int tile_id,
                                                   const uint16_t* __restrict__ blocks,
                                                   const uint16_t* __restrict__ w,
                                                   const int32_t* __restrict__ row_offsets,
                                                   const int32_t* __restrict__ col_indices, uint16_t* __restrict__ out,
                                                   int64_t nnz, int64_t w_rows, int32_t num_row_blocks,
                                                   int32_t d_model, int32_t num_slices, int32_t zero_dead_rows,
                                                   int32_t group) {
  using ML = DmaMainloop<Cfg>;
  constexpr int BM = Cfg::BM, BN = Cfg::BN;
  if (tile_id >= num_row_blocks * num_slices) return;
  const int live_rb = zero_dead_rows ? num_row_blocks : live_row_blocks(row_offsets, num_row_blocks);
  const int tile = xcd_remap(tile_id, live_rb * num_slices);
  int rb, slice;
  tile_coords(tile, live_rb, num_slices, group, &rb, &slice);
  const int n0 = slice * BN;
  int32_t begin = row_offsets[rb];
  int32_t end = row_offsets[rb + 1];
  if (begin < 0 || end > nnz || end < begin) begin = end = 0;  // not a BSR row: treat as empty

  uint16_t* out_tile = out + static_cast<int64_t>(rb) * BM * d_model + n0;
  if (begin == end) {
    if (!zero_dead_rows) return;
    constexpr int kChunksPerRow = BN / 8;
    for (int q = threadIdx.x; q < BM * kChunksPerRow; q += Cfg::kThreads) {
      const int r = q / kChunksPerRow, c = q % kChunksPerRow;
      *reinterpret_cast<u32x4_t*>(out_tile + static_cast<int64_t>(r) * d_model + c * 8) = u32x4_t{0u, 0u, 0u, 0u};
    }
    return;
  }

  DsdDmaSrc<Cfg> src;
  src.blocks = blocks;
  src.w = w + n0;
  src.col_indices = col_indices;
  src.w_rows = w_rows;
  src.d_model = d_model;
  src.begin = begin;
  const ADmaPos<Cfg> ap;
#pragma unroll
  for (int q = 0; q < Cfg::kAInstr; ++q) src.a_off[q] = (ap.row[q] * BM + ap.chunk[q] * 8) * 2u;
  const BDmaPos<Cfg> bp;
#pragma unroll
  for (int q = 0; q < Cfg::kBInstr; ++q)
    src.b_off[q] = (static_cast<uint32_t>(bp.row[q]) * d_model + bp.col[q]) * 2u;

  typename ML::Acc acc;
  ML::run(lds, src, (end - begin) * DsdDmaSrc<Cfg>::kStepsPerBlock, acc);

  // bf16, staged in LDS, then whole row segments per store instruction.
  // Plain stores: the combine reads these rows right away, partly from L2.
  ML::stage_tile(lds, acc, [](float v) { return v; });
  ML::for_each_staged_chunk(lds, [&](int r, int col, u32x4_t v) {
    *reinterpret_cast<u32x4_t*>(out_tile + static_cast<int64_t>(r) * d_model + col) = v;
  });
}

// Two row blocks of BS rows over the same block columns, as one tile of
// 2 BS rows: lane rows past BS read the second row block, `count` blocks on.
// A row block alone: they read zeros (a_off past the buffer).
template <class Cfg, int BS>
struct DsdPairSrc {
  static constexpr int kStepsPerBlock = BS / Cfg::BK;
  static_assert(Cfg::BM == 2 * BS && (!Cfg::APAIR || kStepsPerBlock % 2 == 0), "pairs of row blocks");
  const uint16_t* blocks;
  const uint16_t* w;
  const int32_t* col_indices;
  int64_t w_rows;
  int32_t d_model, begin, count;
  uint32_t a_off[Cfg::kAInstr];
  uint32_t b_off[Cfg::kBInstr];
  __device__ __forceinline__ uint32_t a_voff(int q) const { return a_off[q]; }
  __device__ __forceinline__ uint32_t b_voff(int q) const { return b_off[q]; }
  __device__ __forceinline__ void a_src(int t, __amdgpu_buffer_rsrc_t* r, uint32_t* s) const {
    *r = make_rsrc(blocks + static_cast<int64_t>(begin + t / kStepsPerBlock) * BS * BS,
                   static_cast<uint32_t>(count + 1) * (BS * BS * 2u));
    *s = static_cast<uint32_t>(t % kStepsPerBlock) * (Cfg::BK * 2);
  }
  __device__ __forceinline__ void b_src(int t, __amdgpu_buffer_rsrc_t* r, uint32_t* s) const {
    const int64_t row0 = static_cast<int64_t>(col_indices[begin + t / kStepsPerBlock]) * BS;
    const bool ok = row0 >= 0 && row0 + BS <= w_rows;
    *r = make_rsrc(w + (ok ? row0 : 0) * d_model, ok ? static_cast<uint32_t>(BS) * d_model * 2u : 0u);
    *s = static_cast<uint32_t>(t % kStepsPerBlock) * (Cfg::BK * 2u) * static_cast<uint32_t>(d_model);
  }
};

// Of a row block in a pair, so that both row blocks' offsets fit 32 bits. A row
// block alone (count = 0: the buffer moves on with each block) has no limit.
constexpr int32_t kMaxPairBlocks = 1 << 16;

// Row blocks 2 pair and 2 pair + 1 of BS rows, from column n0 on, by two
// workgroups (which = 0, 1): one tile of 2 BS rows by the first when both
// have the same block columns, else a tile each, its second half of the rows
// empty. Of 64-row blocks, most of a routing layout's are such pairs, and the
// pair's tile reads its columns of w once for both. (One main loop for both
// cases: beside a second one, for tiles of BS rows, the compiler loses the
// ring's stages apart and waits for every load before each step's LDS reads.)
template <class Cfg, int BS>
__device__ __forceinline__ void dsd_pair_tile(uint8_t* __restrict__ lds, int bid, const uint16_t* __restrict__ blocks,
                                              const uint16_t* __restrict__ w,
                                              const int32_t* __restrict__ row_offsets,
                                              const int32_t* __restrict__ col_indices, uint16_t* __restrict__ out,
                                              int64_t nnz, int64_t w_rows, int32_t num_row_blocks, int32_t d_model,
                                              int32_t num_slices, int32_t zero_dead_rows, int32_t group) {
  using ML = DmaMainloop<Cfg>;
  constexpr int BN = Cfg::BN;
  // The second workgroups of all pairs' slices, then the first ones: most of the
  // second ones end at once, and none of them then waits for a CU behind the
  // first ones' tiles (D = 1024, F = 1024, E = 8, 50 row blocks: 0.89 of the time
  // of row blocks one by one, and 1.0 with the second ones last).
  const int pairs = (num_row_blocks + 1) / 2;
  const int which = bid < pairs * num_slices ? 1 : 0;
  const int live_rb = zero_dead_rows ? num_row_blocks : live_row_blocks(row_offsets, num_row_blocks);
  const int live = (live_rb + 1) / 2;
  // A pair's second ones, its slices, one by one over the XCDs: only those of
  // row blocks alone have work, and with all of them on one XCD that needs a
  // round of its own (D = 4096, F = 1024, E = 2, 18 row blocks: 0.83 of the time
  // of row blocks one by one, 1.37 in the order of the first ones).
  const int id = which == 0 ? bid - pairs * num_slices : bid;
  int pair, slice;
  if (which == 0) {
    tile_coords(xcd_remap(id, live * num_slices), live, num_slices, group, &pair, &slice);
  } else {
    pair = uniform(id / num_slices);
    slice = id - pair * num_slices;
  }
  if (pair >= pairs) return;
  const int n0 = slice * BN;
  int rb = 2 * pair;

  // Whether both row blocks have the same columns: all lanes' answer through
  // the ring's LDS (__syncthreads_and would add its own to a full 160 KB).
  bool same = rb + 1 < num_row_blocks;
  if (same) {
    const int32_t b0 = row_offsets[rb], b1 = row_offsets[rb + 1], b2 = row_offsets[rb + 2];
    same = b0 >= 0 && b1 > b0 && b2 <= nnz && b2 - b1 == b1 - b0 && b1 - b0 < kMaxPairBlocks;
    if (same)
      for (int p = threadIdx.x; p < b1 - b0; p += Cfg::kThreads)
        same = same && col_indices[b0 + p] == col_indices[b1 + p];
  }
  int32_t* agree = reinterpret_cast<int32_t*>(lds);
  const bool wave_same = __ballot(!same) == 0;
  if ((threadIdx.x & 63) == 0) agree[threadIdx.x >> 6] = wave_same ? 1 : 0;
  __syncthreads();
  int32_t waves_same = 0;
  for (int v = 0; v < Cfg::kWaves; ++v) waves_same += agree[v];
  const bool both = __builtin_amdgcn_readfirstlane(waves_same) == Cfg::kWaves;
  __syncthreads();
  if (both && which != 0) return;
  if (!both) rb += which;
  if (rb >= num_row_blocks) return;
  int32_t begin = row_offsets[rb];
  int32_t end = row_offsets[rb + 1];
  if (begin < 0 || end > nnz || end < begin) begin = end = 0;  // not a BSR row

  uint16_t* out_tile = out + static_cast<int64_t>(rb) * BS * d_model + n0;
  if (begin == end) {
    if (!zero_dead_rows) return;
    constexpr int kChunksPerRow = BN / 8;
    for (int q = threadIdx.x; q < BS * kChunksPerRow; q += Cfg::kThreads) {
      const int r = q / kChunksPerRow, c = q % kChunksPerRow;
      *reinterpret_cast<u32x4_t*>(out_tile + static_cast<int64_t>(r) * d_model + c * 8) = u32x4_t{0u, 0u, 0u, 0u};
    }
    return;
  }

  DsdPairSrc<Cfg, BS> src;
  src.blocks = blocks;
  src.w = w + n0;
  src.col_indices = col_indices;
  src.w_rows = w_rows;
  src.d_model = d_model;
  src.begin = begin;
  src.count = both ? end - begin : 0;
  const ADmaPos<Cfg> ap;
#pragma unroll
  for (int q = 0; q < Cfg::kAInstr; ++q) {
    const bool second = ap.row[q] >= BS;
    const uint32_t at = (static_cast<uint32_t>(second ? end - begin : 0) * (BS * BS) + (ap.row[q] % BS) * BS +
                         ap.chunk[q] * 8) * 2u;
    src.a_off[q] = second && !both ? kOutOfRange : at;
  }
  const BDmaPos<Cfg> bp;
#pragma unroll
  for (int q = 0; q < Cfg::kBInstr; ++q)
    src.b_off[q] = (static_cast<uint32_t>(bp.row[q]) * d_model + bp.col[q]) * 2u;

  typename ML::Acc acc;
  ML::run(lds, src, (end - begin) * DsdPairSrc<Cfg, BS>::kStepsPerBlock, acc);

  const int rows = both ? 2 * BS : BS;
  ML::stage_tile(lds, acc, [](float v) { return v; });
  ML::for_each_staged_chunk(lds, [&](int r, int col, u32x4_t v) {
    if (r < rows) *reinterpret_cast<u32x4_t*>(out_tile + static_cast<int64_t>(r) * d_model + col) = v;
  });
}

// Which tiles sb_dsd runs: `width` columns (fit_width), deep = the 512-wide
// ones' form for a reduction of at least 8192, paired = block size 64 with the
// row blocks in pairs (dsd_pair_tile).
struct DsdForm {
  int width;
  bool paired, deep;
};

// Block size 64: row blocks one by one, or in pairs. A routing layout
// (`routed`) of E experts has about (row blocks + E) / 2 tile rows in pairs:
// the pairs, and row blocks alone, which cost a whole tile, at every second
// expert's end. Pairs are taken when they let 512-wide tiles that leave CUs
// idle become 256-wide ones (at least 4 row blocks an expert), or when there
// are more tiles than CUs and at least 8 row blocks an expert; the row block
// count may be a worst case, up to E more than there are. But where the pairs
// leave few CUs free, the tiles of row blocks alone may cost a round of their
// own: so the pairs must leave some of the CUs, by the number of experts, or be
// more than one round themselves. Pairs against one by one, F = 1024 and 4096,
// P tiles of pairs on 256 CUs: up to P = 160 0.59-0.92 of the time (1.26 once in
// 211 routings); P = 168-256 0.60-0.92 or, by the routing's chance, 1.06-1.42
// (E = 2 from P = 232 on, E = 4 from 200, E = 8 and 16 from 170); more
// 0.64-0.95. D = 1024, 79 row blocks, E = 20 1.41. D = 4096, 79 row blocks 138
// against 153 us; D = 512 (256 and 128 wide) 29 against 44; 3 row blocks an
// expert (D = 1024, F = 4096, E = 64) 174 against 188.
// Of any other BSR the neighbours' columns differ, and every row block would
// cost a whole tile for its half: none in pairs (64 column blocks, half of
// them in each row: 256 row blocks, D = 1024 129 one by one against 147 us in
// pairs; 64, D = 4096 145 against 160; 16 column blocks, 40 row blocks,
// D = 8192 54 against 67).
inline DsdForm dsd_form(int64_t block_size, int64_t nnz, int64_t w_rows, int64_t num_row_blocks, int64_t d_model,
                        bool routed, int cus) {
  // The reduction depth per row block, from the buffer shape (nnz /
  // num_row_blocks blocks per row).
  const int64_t row_k = nnz / num_row_blocks * block_size;
  const bool deep = row_k >= 8192;
  const int single = fit_width(num_row_blocks, d_model, cus);
  if (block_size != 64 || !routed || row_k <= 0 || row_k >= int64_t{64} * kMaxPairBlocks) return {single, false, deep};
  const int64_t experts = w_rows / row_k;
  const int paired = fit_width((num_row_blocks + experts) / 2, d_model, cus);
  const int64_t least = num_row_blocks - experts;  // row blocks, of a routing layout's worst case
  const int64_t slices = d_model / paired;
  const int eighths = experts <= 2 ? 7 : experts <= 4 ? 6 : 5;
  const bool one_round =
      (num_row_blocks + 1) / 2 * slices <= cus * eighths / 8 && (experts - 1) * slices <= cus / 4;
  const bool rounds = least / 2 * slices > cus;
  const bool narrower = single == 512 && paired == 256 && num_row_blocks >= 4 * experts && one_round;
  const bool many = least * (d_model / single) > cus && num_row_blocks >= 8 * experts && (one_round || rounds);
  if (paired >= 256 && (narrower || many)) return {paired, true, deep};
  return {single, false, deep};
}

}  // namespace sb
