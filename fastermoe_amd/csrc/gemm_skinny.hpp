// Interface of gemm_skinny.hip: the grouped forward product for few rows per expert.
#pragma once
#include "gemm_kernel.hpp"

namespace fmoe {
namespace gemm {

struct SkinnyParams {
    const void *w, *x, *bias;     // [E, n_cols, k], rows of k, [E, n_cols] or null
    void *y, *aux;                // [rows, n_cols]; aux: the pre-activation, or null
    const int32_t *dev_tab;       // segtab layout
    const int64_t *row_index;     // as GemmParams::q_row_index, with its divisor
    int64_t x_total_rows;
    uint32_t div_mul;
    int32_t div_shift;
    int32_t n_cols, k_extent, activation;
    int32_t weights_cached;       // not 0: the weights through the caches, see caches_few_row_weights() in grouped_gemm.hip
    int32_t order_off, tiles_n, extra_groups;   // set by the launch: the table's list of experts (or its map of row tiles), see launch()
};

// rows_cap: the rows that the table was laid out for
int launch_skinny(const SkinnyParams &prm, int dtype, int64_t rows_cap, int64_t n_expert, hipStream_t stream);

}  // namespace gemm
}  // namespace fmoe
