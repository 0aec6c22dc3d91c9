// What the bindings call instead of stir_column_part_hyb_one_sizes where _fill follows on the same stream.
#pragma once
#include <cstdint>

namespace stir {

// Returns when the host has the sizes, or what is wrong with the matrix: the kernel may still be writing the
// workspace.  That may be used, or given back, in the order of the same stream only.
int column_part_hyb_one_sizes(int32_t num_rows, int32_t num_cols, const int32_t* d_indptr, const int32_t* d_indices,
                              int64_t max_nnz, const int32_t* buckets, int32_t num_buckets, void* d_workspace,
                              int64_t* nrows, void* stream, bool whole = false);

}  // namespace stir
