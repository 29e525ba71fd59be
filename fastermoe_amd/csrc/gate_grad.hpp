// Interface of gate_grad.hip for the layer's call (gfx950): the entry points fmoe_gate_weight_grad and fmoe_reduce_slots_gate, for
// 16-bit types also with rows that are no whole 16-byte chunks.
#pragma once
#include "common.hpp"

namespace fmoe {

// whether the two take this gate
bool gate_grad_any_grid(int64_t d_model, int64_t n_expert, int64_t top_k, int dtype);

int gate_weight_grad(const void *grad_score, const int64_t *topk_idx, const void *x, void *grad_w, void *grad_b, int64_t n_tokens,
                     int64_t d_model, int64_t n_expert, int64_t top_k, int dtype, void *workspace, int64_t workspace_bytes, hipStream_t st);

// any_grid: 16-bit rows that are no whole chunks are taken
int reduce_slots_gate(const void *rows, const int64_t *slot_to_row, const void *grad_score, const int64_t *topk_idx, const void *w, void *out,
                      int64_t n_tokens, int64_t top_k, int64_t n_rows, int64_t n_expert, int64_t row_elems, int dtype, bool any_grid, hipStream_t st);

}  // namespace fmoe
