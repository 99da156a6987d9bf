// Residual norms of the final factors (src/Skema_Residuals.hpp:17-217).
#pragma once
#include "sketch.hpp"

namespace skema {

// SVD form: rnorms[c] = ||[A^T u_c - s_c v_c ; A v_c - s_c u_c]||_2, c < r.
// U (m x r), S (r), V (n x r) on the device; rnorms on the host.
void residuals_dense(Ctx* c, int64_t m, int64_t n, int64_t r, const double* A, int64_t lda, const double* U,
                     int64_t ldu, const double* S, const double* V, int64_t ldv, double* rnorms);
void residuals_csr(Ctx* c, int64_t m, int64_t n, int64_t r, int64_t nnz, const int64_t* rowptr, const int32_t* col,
                   const double* val, const double* U, int64_t ldu, const double* S, const double* V, int64_t ldv,
                   double* rnorms);
// A = the n x n Gaussian RBF matrix of the point set (generated by row
// windows, never stored).
void residuals_rbf(Ctx* c, const double* X, int64_t n, int64_t d, int64_t ldp, double gamma, int64_t r,
                   const double* U, int64_t ldu, const double* S, const double* V, int64_t ldv, int64_t window,
                   double* rnorms);
// ||A - U diag(S) V^T||_F^2 += into acc[0] and ||A||_F^2 += into acc[1]
// (device), streamed over row windows of at most w rows.  Caller memory:
// R holds w x n doubles, US w x max(r, 1), part kSumSqPartials; nothing is
// allocated.  Each window adds its two sums to acc in window order.
void residual_fro_stream(hipStream_t st, int64_t m, int64_t n, int64_t r, const double* A, int64_t lda,
                         const double* U, int64_t ldu, const double* S, const double* V, int64_t ldv, int64_t w,
                         double* R, double* US, double* part, double* acc);
// Symmetric (eigenpair) form: rnorms[c] = ||A v_c - s_c v_c||_2.
void residuals_sym_dense(Ctx* c, int64_t n, int64_t r, const double* A, int64_t lda, const double* V, int64_t ldv,
                         const double* S, double* rnorms);
void residuals_sym_csr(Ctx* c, int64_t n, int64_t r, const int64_t* rowptr, const int32_t* col, const double* val,
                       const double* V, int64_t ldv, const double* S, double* rnorms);
void residuals_sym_rbf(Ctx* c, const double* X, int64_t n, int64_t d, int64_t ldp, double gamma, int64_t r,
                       const double* V, int64_t ldv, const double* S, int64_t window, double* rnorms);

}  // namespace skema
