// Row-permute launchers shared between the C ABI (permute.hip) and the fused
// pipeline (pipeline.hip).
#pragma once
#include "common.hpp"

namespace fmoe {

// out[r,:] = inp[index[r] / divisor,:] for r in [0, n_out); rows whose index is
// negative or whose source is outside [0, n_inp) become zero.
int permute_gather_rows(const void *inp, const int64_t *index, int64_t divisor, void *out, int64_t n_out,
                        int64_t n_inp, int64_t row_elems, int dtype, hipStream_t stream);

// out[index[r],:] = inp[r,:] for r in [0, n_in); targets outside [0, n_out) are skipped.
int permute_scatter_rows(const void *inp, const int64_t *index, void *out, int64_t n_in, int64_t n_out,
                         int64_t row_elems, int dtype, hipStream_t stream);

// out[slot_to_row[t top_k + j],:] = inp[t,:] for every token t and choice j; slots without a row in [0, n_out) are skipped, rows
// that no slot names are left alone.  Rows are whole 16-byte chunks and both tensors begin on 16 bytes.
int permute_spread_rows(const void *inp, const int64_t *slot_to_row, int64_t top_k, void *out, int64_t n_tokens, int64_t n_out,
                        int64_t row_elems, int dtype, hipStream_t stream);

// out[r,:] = 0 for every r in [0, n_out) with index[r] < 0.
int permute_zero_unmapped(const int64_t *index, void *out, int64_t n_out, int64_t row_elems, int dtype,
                          hipStream_t stream);

}  // namespace fmoe
