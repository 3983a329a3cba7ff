// The whole MoE layer in one call: routing, SDD + GELU, DSD and combine
// enqueued from native code, every intermediate in one workspace of the
// caller's. A host program that calls the stages one by one pays for the
// arguments, checks and allocations of each (in Python about 50 us for a layer
// whose kernels take 24).
//
// No kernels of its own: each function carves the workspace and calls the
// stages' entry points, so results and checks are theirs.

#include "common.hpp"

namespace sb {
namespace {

constexpr int64_t kBlock = 128;
constexpr int64_t kI32Limit = int64_t{1} << 31;

// Hands out 256-byte aligned pieces of a workspace; with no base it only adds up.
struct Carver {
  uint8_t* base;
  int64_t used = 0;
  template <class T>
  T* take(int64_t count) {
    T* p = base ? reinterpret_cast<T*>(base + used) : nullptr;
    used += (count * static_cast<int64_t>(sizeof(T)) + 255) / 256 * 256;
    return p;
  }
};

// A routing layout (sb_routing's outputs) and the blocks of H and rows of y on it.
struct LayerBuffers {
  int64_t max_row_blocks = 0;
  int32_t *tokens_per_expert, *padded_offsets, *row_token, *copy_row, *row_block_expert, *row_offsets, *col_indices,
      *error;
  uint16_t *h, *y;
};

// The layer kernels take the shape (they address H and one expert's weights
// with 32-bit offsets); others go through sb_sdd and sb_dsd, stage by stage.
int carve_layer(Carver& ws, int64_t num_copies, int64_t num_experts, int64_t d_model, int64_t ffn_dim,
                int64_t max_row_blocks, int64_t max_rows, LayerBuffers* b) {
  if (d_model <= 0 || d_model % 256 != 0 || ffn_dim <= 0 || ffn_dim % 256 != 0)
    return fail(SB_ERR_INVALID, "layer: D and F must be multiples of 256");
  if (max_rows * ffn_dim * 2 >= kI32Limit || ffn_dim * d_model * 2 >= kI32Limit)
    return fail(SB_ERR_INVALID, "layer: H or one expert's weights too large for 32-bit buffer offsets");
  b->max_row_blocks = max_row_blocks;
  b->tokens_per_expert = ws.take<int32_t>(num_experts);
  b->padded_offsets = ws.take<int32_t>(num_experts + 1);
  b->row_token = ws.take<int32_t>(max_rows);
  b->copy_row = ws.take<int32_t>(num_copies);
  b->row_block_expert = ws.take<int32_t>(max_row_blocks);
  b->row_offsets = ws.take<int32_t>(max_row_blocks + 1);
  b->col_indices = ws.take<int32_t>(max_row_blocks * (ffn_dim / kBlock));
  b->error = ws.take<int32_t>(1);
  b->h = ws.take<uint16_t>(max_rows * ffn_dim);
  b->y = ws.take<uint16_t>(max_rows * d_model);
  return SB_OK;
}

// Top-k (num_tokens 0) or assigned routing of num_copies copies.
struct ListBuffers {
  LayerBuffers layer;
  int32_t *counts, *token_offsets, *token_copies;
};

int carve_list(Carver& ws, int64_t num_tokens, int64_t num_copies, int64_t num_experts, int64_t d_model,
               int64_t ffn_dim, ListBuffers* b) {
  int64_t rb = 0, rows = 0, counts = 0;
  if (num_experts <= 0 || num_experts > kI32Limit - 1 || ffn_dim <= 0 || ffn_dim > kI32Limit - 1)
    return fail(SB_ERR_INVALID, "layer: bad expert count or F");
  if (int rc = sb_routing_sizes(num_copies, static_cast<int32_t>(num_experts), static_cast<int32_t>(ffn_dim),
                                static_cast<int32_t>(kBlock), &rb, &rows, &counts))
    return rc;
  if (int rc = carve_layer(ws, num_copies, num_experts, d_model, ffn_dim, rb, rows, &b->layer)) return rc;
  b->counts = ws.take<int32_t>(counts);
  b->token_offsets = ws.take<int32_t>(num_tokens > 0 ? num_tokens + 1 : 0);
  b->token_copies = ws.take<int32_t>(num_tokens > 0 ? num_copies : 0);
  return SB_OK;
}

struct RoundedBuffers {
  LayerBuffers layer;
  int64_t capacity = 0;
  int32_t *scratch, *token_of_copy, *expert_of_copy, *num_assignments, *token_offsets;
  float* weight_of_copy;
};

int carve_rounded(Carver& ws, int64_t num_tokens, int32_t num_experts, int32_t k, int32_t tile, int64_t d_model,
                  int64_t ffn_dim, RoundedBuffers* b) {
  int64_t rb = 0, rows = 0, scratch = 0;
  if (ffn_dim <= 0 || ffn_dim > kI32Limit - 1) return fail(SB_ERR_INVALID, "layer: bad F");
  if (int rc = sb_router_sizes(num_tokens, num_experts, k, tile, static_cast<int32_t>(kBlock),
                               static_cast<int32_t>(ffn_dim), &b->capacity, &rb, &rows, &scratch))
    return rc;
  if (int rc = carve_layer(ws, b->capacity, num_experts, d_model, ffn_dim, rb, rows, &b->layer)) return rc;
  b->scratch = ws.take<int32_t>(scratch);
  b->token_of_copy = ws.take<int32_t>(b->capacity);
  b->expert_of_copy = ws.take<int32_t>(b->capacity);
  b->weight_of_copy = ws.take<float>(b->capacity);
  b->num_assignments = ws.take<int32_t>(1);
  b->token_offsets = ws.take<int32_t>(num_tokens + 1);
  return SB_OK;
}

int check_workspace(const void* workspace, int64_t workspace_bytes, int64_t needed) {
  if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255u) != 0)
    return fail(SB_ERR_INVALID, "layer: the workspace must be 256-byte aligned");
  if (workspace_bytes < needed)
    return fail(SB_ERR_INVALID, "layer: workspace of %lld bytes, %lld needed", static_cast<long long>(workspace_bytes),
                static_cast<long long>(needed));
  return SB_OK;
}

int run_sdd_dsd(const LayerBuffers& b, const void* x, const void* w1, const void* w2, int64_t num_tokens,
                int64_t num_copies, int64_t min_rows, int64_t d_model, int64_t ffn_dim, int64_t num_experts,
                void* stream) {
  if (int rc = sdd_experts(x, w1, b.row_token, b.row_block_expert, b.row_offsets, b.tokens_per_expert,
                           b.padded_offsets, b.h, num_tokens, d_model, ffn_dim, num_experts, b.max_row_blocks, min_rows,
                           1, stream))
    return rc;
  return dsd_experts(b.h, w2, b.tokens_per_expert, b.padded_offsets, b.row_block_expert, b.row_offsets, b.col_indices,
                     b.y, b.max_row_blocks, num_experts, num_copies, min_rows, ffn_dim, d_model, stream);
}

}  // namespace
}  // namespace sb

using namespace sb;

extern "C" int sb_layer_sizes(int64_t num_tokens, int64_t num_copies, int64_t num_experts, int64_t d_model,
                              int64_t ffn_dim, int64_t* workspace_bytes) {
  Carver ws{nullptr};
  ListBuffers b;
  if (int rc = carve_list(ws, num_tokens, num_copies, num_experts, d_model, ffn_dim, &b)) return rc;
  if (workspace_bytes) *workspace_bytes = ws.used;
  return clear_ok();
}

extern "C" int sb_layer_rounded_sizes(int64_t num_tokens, int32_t num_experts, int32_t k, int32_t tile,
                                      int64_t d_model, int64_t ffn_dim, int64_t* workspace_bytes) {
  Carver ws{nullptr};
  RoundedBuffers b;
  if (int rc = carve_rounded(ws, num_tokens, num_experts, k, tile, d_model, ffn_dim, &b)) return rc;
  if (workspace_bytes) *workspace_bytes = ws.used;
  return clear_ok();
}

extern "C" int sb_layer(const void* x, const void* expert_idx, int32_t idx_is_i64, const void* gates,
                        int32_t gate_dtype, const void* w1, const void* w2, void* out, void* workspace,
                        int64_t workspace_bytes, int64_t num_tokens, int32_t k, int32_t num_experts, int64_t d_model,
                        int64_t ffn_dim, const int32_t* valid_tokens, void* stream) {
  if (num_tokens <= 0 || k <= 0 || num_tokens > kI32Limit / k)
    return fail(SB_ERR_INVALID, "expert_idx must be [T, k] with T, k > 0");
  const int64_t n = num_tokens * k;
  Carver ws{static_cast<uint8_t*>(workspace)};
  ListBuffers b;
  if (int rc = carve_list(ws, 0, n, num_experts, d_model, ffn_dim, &b)) return rc;
  if (int rc = check_workspace(workspace, workspace_bytes, ws.used)) return rc;
  const LayerBuffers& l = b.layer;
  if (int rc = sb_routing(expert_idx, idx_is_i64, num_tokens, k, num_experts, static_cast<int32_t>(ffn_dim),
                          static_cast<int32_t>(kBlock), valid_tokens, b.counts, l.tokens_per_expert, l.padded_offsets,
                          l.row_token, l.copy_row, l.row_block_expert, l.row_offsets, l.col_indices, l.error, stream))
    return rc;
  // All copies are routed, but for ids out of range (an error) and tokens from *valid_tokens on.
  const int64_t min_rows = valid_tokens ? 0 : n;
  if (int rc = run_sdd_dsd(l, x, w1, w2, num_tokens, n, min_rows, d_model, ffn_dim, num_experts, stream)) return rc;
  return sb_combine(l.y, l.copy_row, gates, gate_dtype, out, num_tokens, k, d_model, l.max_row_blocks * kBlock,
                    valid_tokens, stream);
}

extern "C" int sb_layer_assigned(const void* x, const void* token_of_copy, int32_t token_is_i64,
                                 const void* expert_of_copy, int32_t expert_is_i64, const void* weights,
                                 int32_t weight_dtype, const void* w1, const void* w2, void* out, void* workspace,
                                 int64_t workspace_bytes, int64_t num_copies, int64_t num_tokens, int32_t num_experts,
                                 int64_t d_model, int64_t ffn_dim, const int32_t* valid_tokens, void* stream) {
  if (num_tokens <= 0 || num_tokens >= kI32Limit - 1) return fail(SB_ERR_INVALID, "routing: bad token count");
  Carver ws{static_cast<uint8_t*>(workspace)};
  ListBuffers b;
  if (int rc = carve_list(ws, num_tokens, num_copies, num_experts, d_model, ffn_dim, &b)) return rc;
  if (int rc = check_workspace(workspace, workspace_bytes, ws.used)) return rc;
  const LayerBuffers& l = b.layer;
  if (int rc = sb_routing_assigned(expert_of_copy, expert_is_i64, token_of_copy, token_is_i64, num_copies, num_tokens,
                                   num_experts, static_cast<int32_t>(ffn_dim), static_cast<int32_t>(kBlock),
                                   valid_tokens, b.counts, l.tokens_per_expert, l.padded_offsets, l.row_token,
                                   l.copy_row, l.row_block_expert, l.row_offsets, l.col_indices, l.error, stream))
    return rc;
  if (int rc = sb_token_csr(token_of_copy, token_is_i64, l.copy_row, num_copies, num_tokens, b.token_offsets,
                            b.token_copies, stream))
    return rc;
  const int64_t min_rows = valid_tokens ? 0 : num_copies;
  if (int rc = run_sdd_dsd(l, x, w1, w2, num_tokens, num_copies, min_rows, d_model, ffn_dim, num_experts, stream))
    return rc;
  return sb_combine_assigned(l.y, l.copy_row, weights, weight_dtype, b.token_offsets, b.token_copies, out, num_tokens,
                             d_model, l.max_row_blocks * kBlock, valid_tokens, stream);
}

extern "C" int sb_layer_rounded(const void* x, const float* scores, const void* w1, const void* w2, void* out,
                                void* workspace, int64_t workspace_bytes, int64_t num_tokens, int32_t num_experts,
                                int32_t k, int32_t tile, int64_t d_model, int64_t ffn_dim, void* stream) {
  Carver ws{static_cast<uint8_t*>(workspace)};
  RoundedBuffers b;
  if (int rc = carve_rounded(ws, num_tokens, num_experts, k, tile, d_model, ffn_dim, &b)) return rc;
  if (int rc = check_workspace(workspace, workspace_bytes, ws.used)) return rc;
  const LayerBuffers& l = b.layer;
  if (int rc = sb_token_rounding(scores, num_tokens, num_experts, k, tile, static_cast<int32_t>(kBlock),
                                 static_cast<int32_t>(ffn_dim), b.scratch, b.token_of_copy, b.expert_of_copy,
                                 b.weight_of_copy, b.num_assignments, b.token_offsets, l.tokens_per_expert,
                                 l.padded_offsets, l.row_token, l.copy_row, l.row_block_expert, l.row_offsets,
                                 l.col_indices, l.error, stream))
    return rc;
  // Rounding, to the tile or the largest multiple of it in T, takes less than a tile from an expert.
  const int64_t min_rows = num_tokens * k - static_cast<int64_t>(num_experts) * (tile - 1);
  if (int rc = run_sdd_dsd(l, x, w1, w2, num_tokens, b.capacity, min_rows, d_model, ffn_dim, num_experts, stream))
    return rc;
  return sb_combine_assigned(l.y, l.copy_row, b.weight_of_copy, SB_DTYPE_F32, b.token_offsets, nullptr, out,
                             num_tokens, d_model, l.max_row_blocks * kBlock, nullptr, stream);
}
