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
    int32_t n_cols, k_extent, tiles_n, map_off, activation;
};
constexpr int kSkinnyCols = 16;   // columns of a workgroup

// row_tiles: the most 128-row tiles the table can have
int launch_skinny(const SkinnyParams &prm, int dtype, int64_t row_tiles, hipStream_t stream);

}  // namespace gemm
}  // namespace fmoe
