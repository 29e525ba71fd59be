// A whole layer pass -- gate, routing, experts, combine, or their backward -- enqueued by one call (gfx950).
//
// Host code only: the entry points that the layer otherwise calls one by one, in the same order on the same
// stream.  A decoding step is five kernels of 3 to 9 us, which Python, the bindings and autograd took 100 us to enqueue one
// by one; a training step of 2000 rows is sixteen in 270 us, enqueued in 390.
//
// All intermediate tensors of a pass lie in one scratch block of the caller's, or, where the backward needs them, in
// tensors that it hands in.  Blocks whose lives do not overlap share memory: the sorted input is the output rows' place before the
// second linear writes them, and in the backward one block of rows is in turn the gradient of the experts' output, the
// experts' input gradient and the sorted input.
#include "gate_grad.hpp"
#include "grouped_gemm.hpp"
#include "permute.hpp"

#include <algorithm>
#include <cstdlib>
#include <cstring>

namespace fmoe {
namespace {

struct Sizes {
    int64_t n_tokens, d_model, d_hidden, n_expert, top_k, n_slots;
    int dtype, activation, eb;
};

bool switched_off(const char *name) {
    const char *v = getenv(name);
    return v != nullptr && !strcmp(v, "0");
}

// Consecutive 256-byte aligned pieces of a block; without a base it only adds up.
struct Carver {
    unsigned char *base;
    int64_t used = 0;
    void *take(int64_t bytes) {
        void *p = base ? base + used : nullptr;
        used += (bytes + 255) / 256 * 256;
        return p;
    }
};

// whether rows are whole 16-byte chunks; where they are not, 16-bit types go through gemm_unaligned.hip, over sorted rows
bool on_grid(const Sizes &s) { return fmoe_linear_dev_supported(s.d_model, s.d_hidden, s.dtype) == 1; }

bool reads_token_rows(const Sizes &s, bool keep_pre) {
    return on_grid(s) && s.n_tokens * s.d_model * s.eb < ((int64_t)1 << 31) &&
           !fmoe_linear_act_dev_reads_rows(s.n_slots, s.n_expert, s.d_model, s.d_hidden, s.dtype, s.activation, keep_pre);
}

int64_t split_bytes(int64_t contraction, int dtype, int64_t bytes) {
    return switched_off("FMOE_DEV_SPLIT") || fmoe_linear_dev_workspace_bytes(contraction, dtype) == 0 ? 0 : bytes;
}

struct Forward {   // scratch of a forward
    int64_t *counts;
    void *route_ws, *split_ws;
    int64_t route_bytes, split1, split2;
    // where nothing is kept for a backward
    int64_t *idx, *pos, *s2r;
    void *score, *table, *mid, *rows;
};
Forward forward_layout(const Sizes &s, bool keep, int gate, Carver &c) {
    Forward f{};
    const bool keep_pre = keep && s.activation == FMOE_ACT_GELU;
    if (gate != FMOE_GATE_ROUTED) {
        f.counts = (int64_t *)c.take(s.n_expert * 8);
        f.route_bytes = fmoe_routing_workspace_bytes(s.n_slots, s.n_expert);
        f.route_ws = c.take(f.route_bytes);
    }
    f.split1 = split_bytes(s.d_model, s.dtype, fmoe_linear_forward_dev_workspace_bytes(
        s.n_slots, s.n_expert, s.d_model, s.d_hidden, s.dtype, s.activation, keep_pre, reads_token_rows(s, keep_pre)));
    f.split2 = split_bytes(s.d_hidden, s.dtype, fmoe_linear_forward_dev_workspace_bytes(
        s.n_slots, s.n_expert, s.d_hidden, s.d_model, s.dtype, FMOE_ACT_NONE, 0, 0));
    f.split_ws = c.take(std::max(f.split1, f.split2));
    if (!keep) {
        if (gate != FMOE_GATE_ROUTED) {
            f.idx = (int64_t *)c.take(s.n_slots * 8);
            f.score = c.take(s.n_slots * s.eb);
            f.pos = (int64_t *)c.take(s.n_slots * 8);
            f.s2r = (int64_t *)c.take(s.n_slots * 8);
            f.table = c.take(fmoe_segment_table_bytes(s.n_slots, s.n_expert));
        }
        f.mid = c.take(s.n_slots * s.d_hidden * s.eb);
        f.rows = c.take(s.n_slots * s.d_model * s.eb);
    }
    return f;
}

struct Backward {   // scratch of a backward
    void *rows, *grad_pre, *grad_score, *ws;
    int64_t split2, split1, gate_bytes;
};
Backward backward_layout(const Sizes &s, int gate, Carver &c) {
    Backward b{};
    b.rows = c.take(s.n_slots * s.d_model * s.eb);
    b.grad_pre = c.take(s.n_slots * s.d_hidden * s.eb);
    b.split2 = split_bytes(s.d_model, s.dtype, fmoe_linear_dgrad_dev_workspace_bytes(s.n_slots, s.n_expert, s.d_hidden, s.d_model,
                                                                                   s.dtype, s.activation));
    b.split1 = split_bytes(s.d_hidden, s.dtype, fmoe_linear_dgrad_dev_workspace_bytes(s.n_slots, s.n_expert, s.d_model, s.d_hidden,
                                                                                    s.dtype, FMOE_ACT_NONE));
    if (gate != FMOE_GATE_ROUTED) {
        b.grad_score = c.take(s.n_slots * s.eb);
        b.gate_bytes = fmoe_gate_weight_grad_workspace_bytes(s.n_tokens, s.d_model, s.n_expert);
    }
    b.ws = c.take(std::max({b.split1, b.split2, b.gate_bytes}));
    return b;
}

bool taken(const Sizes &s, int gate) {
    if (s.n_tokens < 1 || s.d_model < 1 || s.d_hidden < 1 || s.n_expert < 1 || s.top_k < 1 || s.eb == 0 || s.dtype == FMOE_F64) return false;
    if (s.n_tokens > (int64_t)INT32_MAX / s.top_k - 65536 || s.n_expert > (1 << 24)) return false;
    if (s.activation < FMOE_ACT_NONE || s.activation > FMOE_ACT_GELU) return false;
    if (!on_grid(s) && (s.dtype == FMOE_F32 || s.d_model * s.eb > (1 << 22) || s.d_hidden * s.eb > (1 << 22))) return false;
    if (gate == FMOE_GATE_ROUTED) return true;
    if (gate == FMOE_GATE_LINEAR && !fmoe_gate_grad_supported(s.d_model, s.n_expert, s.top_k, s.dtype)) return false;
    if (gate == FMOE_GATE_LINEAR) return fmoe_gate_linear_supported(s.d_model, s.n_expert, s.top_k, s.dtype) == 1;
    return gate == FMOE_GATE_LOGITS && (s.top_k == 1 || s.top_k == 2 || s.top_k == 4 || s.top_k == 8) && s.top_k <= s.n_expert && s.n_expert <= 8192;
}

// the switches that keep the steps of a layer apart
bool apart(int gate) {
    return switched_off("FMOE_FOLD_COMBINE") || switched_off("FMOE_EXPERT_EPILOGUE") || switched_off("FMOE_DEVICE_TABLES") ||
           (gate != FMOE_GATE_ROUTED && switched_off("FMOE_GATE_LINEAR_FUSED"));
}

// The sorted copy of the token rows.  Rows past the routed ones are left alone: the products read the segments of the table only.
int sort_rows(const Sizes &s, const void *x, const int64_t *pos, const int64_t *slot_to_row, void *rows, hipStream_t st) {
    if (s.top_k > 1 && s.d_model * s.eb % 16 == 0 && aligned16(x) && aligned16(rows))
        return permute_spread_rows(x, slot_to_row, s.top_k, rows, s.n_tokens, s.n_slots, s.d_model, s.dtype, st);
    return permute_gather_rows(x, pos, s.top_k, rows, s.n_slots, s.n_tokens, s.d_model, s.dtype, st);
}

// one expert linear over the sorted rows of a segment table
int linear_forward(const Sizes &s, const void *x, const int64_t *row_index, const void *w, const void *b, void *pre, void *y,
                   const void *table, int64_t in_feat, int64_t out_feat, int activation, bool keep, void *ws, int64_t ws_bytes, hipStream_t st) {
    const bool plain = activation == FMOE_ACT_NONE && pre == nullptr;
    LinearForwardArgs a{x, w, b, y, pre, in_feat, out_feat, s.dtype, plain ? kEpiStore : kEpiBiasAct, activation};
    a.x_row_index = row_index;
    a.x_index_div = row_index ? s.top_k : 1;
    a.x_total_rows = row_index ? s.n_tokens : 0;
    a.dev_tab = (const int32_t *)table;
    a.dev_rows_cap = s.n_slots;
    a.dev_workspace = ws_bytes ? ws : nullptr;
    a.dev_workspace_bytes = ws_bytes;
    a.dev_any_grid = true;
    a.dev_weights_once = !keep;
    return grouped_linear_forward(a, nullptr, s.n_expert, 0, s.n_slots, st);
}
int linear_dgrad(const Sizes &s, const void *gy, const void *w, const void *pre, void *gx, const void *table, int64_t in_feat,
                 int64_t out_feat, int activation, void *ws, int64_t ws_bytes, hipStream_t st) {
    const bool act = activation != FMOE_ACT_NONE;
    LinearDgradArgs d{gy, w, gx, act ? pre : nullptr, in_feat, out_feat, s.dtype, act ? kEpiDAct : kEpiStore, activation};
    d.dev_tab = (const int32_t *)table;
    d.dev_rows_cap = s.n_slots;
    d.dev_workspace = ws_bytes ? ws : nullptr;
    d.dev_workspace_bytes = ws_bytes;
    d.dev_any_grid = true;
    return grouped_linear_dgrad(d, nullptr, s.n_expert, 0, s.n_slots, st);
}
int linear_wgrad(const Sizes &s, const void *gy, const void *x, void *gw, void *gb, const void *table, int64_t in_feat, int64_t out_feat,
                 hipStream_t st) {
    LinearWgradArgs g{gy, x, gw, gb, in_feat, out_feat, s.dtype};
    g.dev_tab = (const int32_t *)table;
    g.dev_rows_cap = s.n_slots;
    g.dev_any_grid = true;
    return grouped_linear_wgrad(g, nullptr, s.n_expert, 0, s.n_slots, true, st);
}

Sizes sizes_of(int64_t n_tokens, int64_t d_model, int64_t d_hidden, int64_t n_expert, int64_t top_k, int dtype, int activation) {
    return Sizes{n_tokens, d_model, d_hidden, n_expert, top_k, n_tokens > 0 && top_k > 0 ? n_tokens * top_k : 0, dtype, activation,
                 dtype_bytes(dtype)};
}

}  // namespace
}  // namespace fmoe

using namespace fmoe;

extern "C" int fmoe_layer_sizes(int64_t n_tokens, int64_t d_model, int64_t d_hidden, int64_t n_expert, int64_t top_k, int dtype,
                                int activation, int keep, int gate, int64_t *sizes_host) {
    const Sizes s = sizes_of(n_tokens, d_model, d_hidden, n_expert, top_k, dtype, activation);
    if (!taken(s, gate) || sizes_host == nullptr) return 0;
    Carver fwd{nullptr}, bwd{nullptr};
    forward_layout(s, keep != 0, gate, fwd);
    sizes_host[0] = fwd.used;
    sizes_host[1] = 0;
    if (keep) {
        backward_layout(s, gate, bwd);
        sizes_host[1] = bwd.used;
    }
    sizes_host[2] = fmoe_segment_table_bytes(s.n_slots, s.n_expert);
    return apart(gate) ? 0 : 1;
}

extern "C" int fmoe_layer_forward(const void *x, const void *gate_w, const void *gate_b, const void *logits, const void *w1,
                                  const void *b1, const void *w2, const void *b2, int64_t *topk_idx, void *topk_score, int64_t *pos,
                                  int64_t *slot_to_row, void *segment_table, void *pre, void *mid, void *rows, void *out,
                                  int64_t n_tokens, int64_t d_model, int64_t d_hidden, int64_t n_expert, int64_t top_k, int dtype,
                                  int activation, int keep, int gate, void *scratch, int64_t scratch_bytes, void *stream) {
    const Sizes s = sizes_of(n_tokens, d_model, d_hidden, n_expert, top_k, dtype, activation);
    FMOE_REQUIRE(taken(s, gate), "fmoe_layer_forward: n_tokens=%lld d_model=%lld d_hidden=%lld n_expert=%lld top_k=%lld dtype=%d is not taken",
                 (long long)n_tokens, (long long)d_model, (long long)d_hidden, (long long)n_expert, (long long)top_k, dtype);
    Carver c{(unsigned char *)scratch};
    const Forward f = forward_layout(s, keep != 0, gate, c);
    if (scratch_bytes < c.used || (scratch == nullptr && c.used > 0) || !aligned16(scratch))
        return fail(FMOE_EWORKSPACE, "fmoe_layer_forward: needs %lld bytes of 16-byte aligned scratch, got %lld", (long long)c.used,
                    (long long)scratch_bytes);
    if (!keep) {
        if (gate != FMOE_GATE_ROUTED) { topk_idx = f.idx; topk_score = f.score; pos = f.pos; slot_to_row = f.s2r; segment_table = f.table; }
        mid = f.mid; rows = f.rows;
    }
    const bool keep_pre = keep && activation == FMOE_ACT_GELU;
    FMOE_REQUIRE(x && w1 && w2 && topk_score && pos && slot_to_row && segment_table && mid && rows && out && (gate == FMOE_GATE_ROUTED || topk_idx) &&
                     (pre || !keep_pre), "fmoe_layer_forward: NULL pointer");
    const int64_t table_bytes = fmoe_segment_table_bytes(s.n_slots, n_expert);
    int rc = FMOE_OK;
    if (gate == FMOE_GATE_LINEAR)
        rc = fmoe_gate_linear_topk_route_table(x, gate_w, gate_b, n_tokens, d_model, n_expert, top_k, dtype, 0, topk_idx, topk_score, f.counts,
                                               pos, slot_to_row, segment_table, table_bytes, f.route_ws, f.route_bytes, stream);
    else if (gate == FMOE_GATE_LOGITS)
        rc = fmoe_gate_topk_route_table(logits, n_tokens, n_expert, top_k, dtype, 0, topk_idx, topk_score, f.counts, pos, slot_to_row,
                                        segment_table, table_bytes, f.route_ws, f.route_bytes, stream);
    if (rc != FMOE_OK) return rc;
    const bool token_rows = reads_token_rows(s, keep_pre);
    if (!token_rows) {
        rc = sort_rows(s, x, pos, slot_to_row, rows, (hipStream_t)stream);
        if (rc != FMOE_OK) return rc;
    }
    hipStream_t st = (hipStream_t)stream;
    rc = linear_forward(s, token_rows ? x : rows, token_rows ? pos : nullptr, w1, b1, keep_pre ? pre : nullptr, mid, segment_table, d_model,
                        d_hidden, activation, keep != 0, f.split_ws, f.split1, st);
    if (rc != FMOE_OK) return rc;
    rc = linear_forward(s, mid, nullptr, w2, b2, nullptr, rows, segment_table, d_hidden, d_model, FMOE_ACT_NONE, keep != 0, f.split_ws, f.split2, st);
    if (rc != FMOE_OK) return rc;
    return fmoe_gather_combine_forward(rows, slot_to_row, topk_score, out, n_tokens, top_k, s.n_slots, d_model, dtype, stream);
}

extern "C" int fmoe_layer_backward(const void *grad_out, const void *x, const void *gate_w, const void *w1, const void *w2,
                                   const int64_t *topk_idx, const void *topk_score, const int64_t *pos, const int64_t *slot_to_row,
                                   const void *segment_table, const void *pre, const void *mid, const void *rows, void *grad_x,
                                   void *grad_score, void *grad_gate_w, void *grad_gate_b, void *grad_w1, void *grad_b1, void *grad_w2,
                                   void *grad_b2, int64_t n_tokens, int64_t d_model, int64_t d_hidden, int64_t n_expert, int64_t top_k,
                                   int dtype, int activation, int gate, void *scratch, int64_t scratch_bytes, void *stream) {
    const Sizes s = sizes_of(n_tokens, d_model, d_hidden, n_expert, top_k, dtype, activation);
    FMOE_REQUIRE(taken(s, gate), "fmoe_layer_backward: n_tokens=%lld d_model=%lld d_hidden=%lld n_expert=%lld top_k=%lld dtype=%d is not taken",
                 (long long)n_tokens, (long long)d_model, (long long)d_hidden, (long long)n_expert, (long long)top_k, dtype);
    Carver c{(unsigned char *)scratch};
    const Backward b = backward_layout(s, gate, c);
    if (scratch_bytes < c.used || scratch == nullptr || !aligned16(scratch))
        return fail(FMOE_EWORKSPACE, "fmoe_layer_backward: needs %lld bytes of 16-byte aligned scratch, got %lld", (long long)c.used,
                    (long long)scratch_bytes);
    const bool gated = gate != FMOE_GATE_ROUTED;
    if (gated) grad_score = b.grad_score;
    const void *saved_pre = activation == FMOE_ACT_GELU ? pre : mid;   // (ReLU's derivative can be read off its output)
    FMOE_REQUIRE(grad_out && x && w1 && w2 && topk_score && pos && slot_to_row && segment_table && saved_pre && mid && rows && grad_score &&
                     (!gated || (topk_idx && gate_w)), "fmoe_layer_backward: NULL pointer");
    // (what the gate's kernels would refuse, before anything is enqueued)
    if (gated && grad_gate_w != nullptr && !gate_grad_any_grid(d_model, n_expert, top_k, dtype))
        return fail(FMOE_ELIMIT, "fmoe_layer_backward: gradients of a gate of d_model=%lld n_expert=%lld top_k=%lld dtype=%d are not taken",
                    (long long)d_model, (long long)n_expert, (long long)top_k, dtype);
    FMOE_REQUIRE(!gated || grad_x == nullptr || (aligned16(gate_w) && aligned16(grad_x)), "fmoe_layer_backward: misaligned gate_w or grad_x");
    FMOE_REQUIRE(!gated || grad_gate_w == nullptr || aligned16(x), "fmoe_layer_backward: misaligned x");
    hipStream_t st = (hipStream_t)stream;
    int rc = fmoe_gather_combine_backward(grad_out, rows, slot_to_row, topk_score, b.rows, grad_score, n_tokens, top_k, s.n_slots, d_model,
                                          dtype, stream);
    if (rc != FMOE_OK) return rc;
    const bool first = grad_x != nullptr || grad_w1 != nullptr;   // whether the first linear's output gradient is wanted
    if (first) {
        rc = linear_dgrad(s, b.rows, w2, saved_pre, b.grad_pre, segment_table, d_hidden, d_model, activation, b.ws, b.split2, st);
        if (rc != FMOE_OK) return rc;
    }
    if (grad_w2 != nullptr) {
        rc = linear_wgrad(s, b.rows, mid, grad_w2, grad_b2, segment_table, d_hidden, d_model, st);
        if (rc != FMOE_OK) return rc;
    }
    if (grad_x != nullptr) {
        rc = linear_dgrad(s, b.grad_pre, w1, nullptr, b.rows, segment_table, d_model, d_hidden, FMOE_ACT_NONE, b.ws, b.split1, st);
        if (rc != FMOE_OK) return rc;
        // (the gate's part of the input gradient is added in the same pass, before the one rounding)
        rc = gated ? reduce_slots_gate(b.rows, slot_to_row, grad_score, topk_idx, gate_w, grad_x, n_tokens, top_k, s.n_slots, n_expert,
                                       d_model, dtype, true, st)
                   : fmoe_reduce_slots(b.rows, slot_to_row, grad_x, n_tokens, top_k, s.n_slots, d_model, dtype, stream);
        if (rc != FMOE_OK) return rc;
    }
    if (grad_w1 != nullptr) {
        rc = sort_rows(s, x, pos, slot_to_row, b.rows, st);
        if (rc != FMOE_OK) return rc;
        rc = linear_wgrad(s, b.grad_pre, b.rows, grad_w1, grad_b1, segment_table, d_model, d_hidden, st);
        if (rc != FMOE_OK) return rc;
    }
    if (gated && grad_gate_w != nullptr)
        rc = gate_weight_grad(grad_score, topk_idx, x, grad_gate_w, grad_gate_b, n_tokens, d_model, n_expert, top_k, dtype, b.ws,
                              b.gate_bytes, st);
    return rc;
}
