// The layer kernels' tile schedules, compiled for the CPU: extern "C" shims
// over the same __host__ __device__ functions the kernels call
// (common.hpp: xcd_remap, split_tail, split_tail_slack, tile_coords;
// dsd_tile.hpp: dsd_form; sdd_tile.hpp: sdd_form;
// expert_chunks.hpp: balanced_chunk_tile, lpt_group_tile, pair_units_per_xcd,
// pair_tile_for, narrow_width, may_be_narrow, narrow_tile_for), so
// tests/test_tile_schedules.py and tests/test_narrow_tiles.py check the
// compiled mappings themselves. Part of the tool library (libsparsebench_probe.so),
// not of libsparsebench_hip.so's C ABI. No kernel runs.

#include "dsd_tile.hpp"
#include "expert_chunks.hpp"
#include "sdd_tile.hpp"

using namespace sb;

// sb_dsd's form (dsd_tile.hpp): width + 1 if in pairs + 2 if deep.
extern "C" int sbt_dsd_form(int64_t block_size, int64_t nnz, int64_t w_rows, int64_t num_row_blocks, int64_t d_model,
                            int routed, int cus) {
  const DsdForm f = dsd_form(block_size, nnz, w_rows, num_row_blocks, d_model, routed != 0, cus);
  return f.width + (f.paired ? 1 : 0) + (f.deep ? 2 : 0);
}

extern "C" int sbt_sdd_form(int64_t num_row_blocks, int64_t d_model, int64_t ffn_dim, int cus) {
  return static_cast<int>(sdd_form(num_row_blocks, d_model, ffn_dim, cus));
}

extern "C" int sbt_xcd_remap(int bid, int live) { return xcd_remap(bid, live); }

extern "C" void sbt_split_tail(int bid, int tiles, int cus_per_xcd, int* tile, int* half) {
  const TailTile t = split_tail(bid, tiles, cus_per_xcd);
  *tile = t.tile;
  *half = t.half;
}

extern "C" int64_t sbt_split_tail_slack(int cus) { return split_tail_slack(cus); }

extern "C" void sbt_tile_coords(int tile, int live_rb, int slices, int group, int* rb, int* slice) {
  tile_coords(tile, live_rb, slices, group, rb, slice);
}

extern "C" int sbt_balanced_chunk_tile(int bid, int chunks, int slices, int* rank, int* slice) {
  return balanced_chunk_tile(bid, chunks, slices, rank, slice) ? 1 : 0;
}

extern "C" int sbt_pair_units_per_xcd(int units) { return pair_units_per_xcd(units); }

extern "C" int sbt_pair_tile_for(int bid, int pairs, int singles, int slices, int cus, int* single, int* k,
                                 int* slice, int* half) {
  bool s = false;
  const bool ok = pair_tile_for(bid, pairs, singles, slices, cus, &s, k, slice, half);
  *single = s ? 1 : 0;
  return ok ? 1 : 0;
}

extern "C" void sbt_lpt_group_tile(int local, int groups, int slices, uint32_t big, int* pos, int* slice) {
  lpt_group_tile(local, groups, slices, big, pos, slice);
}

extern "C" int sbt_narrow_width(int live_rb, int columns, int widest, int cus) {
  return narrow_width(live_rb, columns, widest, cus);
}

extern "C" int sbt_may_be_narrow(int64_t min_rows, int64_t columns, int widest, int cus) {
  return may_be_narrow(min_rows, columns, widest, cus) ? 1 : 0;
}

extern "C" void sbt_narrow_tile_for(int bid, int live_rb, int slices, int* rb, int* slice) {
  narrow_tile_for(bid, live_rb, slices, rb, slice);
}
