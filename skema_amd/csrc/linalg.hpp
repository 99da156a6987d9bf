// FP64 dense linear algebra used by the fixed-rank finalize
// (reference: linalg::qr / ls / svd in src/Skema_BlasLapack.hpp:71-243).
#pragma once
#include <vector>

#include "common.hpp"
#include "gemm.hpp"

namespace skema {

// Householder QR with LAPACK dgeqr2 conventions (dlarfg: beta =
// -sign(alpha)*||x||, tau = (beta-alpha)/beta, v(0) = 1).  On return A (m x n,
// m >= n, leading dimension lda) holds R on and above the diagonal and the
// reflectors below it; tau has n entries.  Blocked like dgeqrf: panels of 32
// columns are factored column by column (one launch for a panel of at most
// 1024 rows, one launch per column with the rows spread over the CUs
// otherwise) and their compact WY form I - V T V^T is applied to the trailing
// columns with FP64 MFMA GEMMs.  The T factors stay in the workspace.  thin_qr
// takes this for matrices whose panels cannot be factored by products.
void householder_qr(hipStream_t st, int64_t m, int64_t n, double* A, int64_t lda, double* tau, DevBuf* work,
                    GemmWorkspace* gws);

// Explicit thin Q (m x n) from the reflectors left in A by householder_qr
// (dorgqr semantics: each panel's I - V T V^T applied to [I; 0] by GEMMs, last
// panel first), with the T factors householder_qr left in `work` (A was the
// last matrix factored with this workspace).  Q must not alias A.
void householder_q(hipStream_t st, int64_t m, int64_t n, const double* A, int64_t lda, double* Q, int64_t ldq,
                   DevBuf* work, GemmWorkspace* gws);

// Thin Q (m x n) and, where R is not null, R (n x n) of A (m x n, m >= n,
// overwritten) with the signs of householder_qr, its panels factored by
// products (qr_panel.hip).  False when a panel's columns are too dependent for
// that (or not finite), or one has nothing below its diagonal (its sign is not the
// products' to pick): A, Q and R then hold nothing of use.  Waits for the stream.
bool thin_qr_products(hipStream_t st, int64_t m, int64_t n, double* A, int64_t lda, double* Q, int64_t ldq, double* R,
                      int64_t ldr, DevBuf* work, GemmWorkspace* gws);

// R (n x n, upper, zero below) from the factored A.
void extract_r(hipStream_t st, int64_t n, const double* A, int64_t lda, double* R, int64_t ldr);

// Whether the panel products take less time than the column by column form: not
// for a few columns, where their five launches and the wait for their flag cost
// more than a launch a column, or, up to 1024 rows, one launch for all columns,
// whose time grows with the rows.  The factors of a 5000 x 300 sketch by products
// -> column by column: range 1 791 -> 423 us, range 5 964 -> 728, range 8
// 1158 -> 976; range 9 983 by products.
inline bool panel_products_pay(int64_t m, int64_t n) { return n > 8 || (m > 512 && m <= 1024) || m > 32768; }

// The same for any A: `load` writes the matrix into A (again, to be factored
// with householder_qr, where the products gave up).  tau: n entries of scratch.
template <class Load>
void thin_qr(hipStream_t st, int64_t m, int64_t n, double* A, int64_t lda, double* Q, int64_t ldq, double* R, int64_t ldr,
             double* tau, DevBuf* work, GemmWorkspace* gws, Load&& load) {
  load();
  if (panel_products_pay(m, n)) {
    if (thin_qr_products(st, m, n, A, lda, Q, ldq, R, ldr, work, gws)) return;
    load();
  }
  householder_qr(st, m, n, A, lda, tau, work, gws);
  if (R) extract_r(st, n, A, lda, R, ldr);
  householder_q(st, m, n, A, lda, Q, ldq, work, gws);
}

// B <- T^{-1} B for upper-triangular T (n x n), B (n x nrhs).  This is what
// dgels('N') reduces to when its input is already upper triangular.
void trsm_upper(hipStream_t st, int64_t n, int64_t nrhs, const double* T, int64_t ldt, double* B,
                int64_t ldb);

// B (cols x rows) <- A^T for A (rows x cols).
void transpose(hipStream_t st, int64_t rows, int64_t cols, const double* A, int64_t lda, double* B,
               int64_t ldb);

// One-sided Jacobi SVD of a square n x n matrix A (overwritten).  Produces
// U (n x n), S (n, descending) and V (n x n) with A = U diag(S) V^T.
// Returns the number of sweeps used; throws kErrNumeric when pairs still
// rotate after 100 sweeps.
int jacobi_svd(hipStream_t st, int64_t n, double* A, int64_t lda, double* U, int64_t ldu, double* S,
               double* V, int64_t ldv, DevBuf* scratch);

}  // namespace skema
