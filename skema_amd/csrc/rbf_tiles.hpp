// FP64 products with rows of the Gaussian RBF matrix of a point set.
#pragma once
#include "gemm.hpp"
#include "sketch.hpp"

namespace skema {

constexpr int kRbfMaxFeat = 128;  // features of the Gram form (more: direct differences, rbf.hip)

// Rows [row0, row0 + rows) of K = exp(-gamma ||x_i - x_j||^2) over n points.
struct RbfRows {
  const double* X = nullptr;  // points, n x d column-major
  int64_t n = 0, ldp = 0, d = 0;
  const double* nrm = nullptr;  // ||x_j||^2, n entries
  double gamma = 0.0;
  int64_t row0 = 0, rows = 0;
};

// With K's rows formed once, a range of points at a time in c->kwin:
//   U != null : left  (k x n) through `left`, U (k x rows, ldu) K
//   OP != null: right (rows x N) through `right`, K OP^T with OP N x n (ldop)
// (both outputs per their alpha and beta, columns of `right` split as in
// gemm_f64).  `timed`: event names "window", "rbf_left" and "rbf_right".
void rbf_products_f64(Ctx* c, const RbfRows& w, const double* U, int64_t ldu, int64_t k, const GemmOut& left,
                      const double* OP, int64_t ldop, int64_t N, const GemmOut& right, bool timed);

// C (rows x cols, ldc): K(row0 + i, col0 + j); when part is not null, C <-
// 2 C o K in place and part[b] = sum over a block of (its 2 C o K) o D, counted
// twice for columns j >= twice.  Returns the number of blocks (entries of part).
int64_t rbf_tile_blocks(int64_t rows, int64_t cols);
void rbf_tiles_f64(hipStream_t st, const RbfRows& w, int64_t col0, int64_t cols, double* C, int64_t ldc, int64_t twice,
                   double* part);

// Grow-only scratch for a rows x n panel cut to `unit` columns or more: the
// most columns (a multiple of unit, at most n rounded up) that fit `most` bytes,
// less where the device has no room.
int64_t reserve_columns(DevBuf& buf, int64_t ld, int64_t n, int64_t unit, size_t most);

bool rbf_tiles_supported(const Sketch& sk);
// have_norms: sk.win holds this point set's norms (a later window of one
// linear_update).
void update_rbf_window_tiles(Sketch& sk, const double* points, int64_t ldp, int64_t row0, int64_t rows, bool have_norms);

}  // namespace skema
