// Whole-matrix pass of linear_update over CSR input (closed form of the
// window recurrence from a zero state; see csr_pass.hip).
#pragma once
#include "sketch.hpp"

namespace skema {

// Columns a tile of the left product over m x n entries with na map rows in all;
// 0: the column by column form.
int64_t left_tile_cols(int64_t m, int64_t n, int64_t na);

// What the pass keeps of a sketch's sparse maps (Sketch::ell_pair).
void prepare_csr_maps(Sketch& sk);

// nnz: the nonzeros, as inspect_csr found them.
void update_csr_all(Sketch& sk, const int64_t* rowptr, const int32_t* col, const double* val, int64_t nnz);

}  // namespace skema
