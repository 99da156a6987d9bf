// Thin QR (Q and R of a tall FP64 matrix) with panels of 32 columns factored
// by products instead of column by column.
//
// Householder QR needs one reduction over the rows per column; a panel of 32
// took 33 dependent launches (21 us each at 65536 rows).  Here a panel P goes
// through the matrix cores five times:
//   G1 = P^T P,  G1 = R1^T R1             (Cholesky)
//   Q1 = P R1^{-1},  G2 = Q1^T Q1 = R2^T R2
//   Q  = Q1 R2^{-1}, R' = R2 R1           (Cholesky QR twice: Q orthonormal to eps;
//                                          Yamamoto, Nakatsukasa, Yanagisawa, Fukaya 2015)
// and the reflectors follow from Q: with D the signs LAPACK's dlarfg would pick
// (R = D R', R_jj = -sign(a_jj) |.|), Q D - [I; 0] = V U with V unit lower
// trapezoidal and U upper triangular, an LU factorisation without pivoting whose
// pivots lie in [-2, -1] because D_j is picked against the sign of the pivot
// (Householder vectors from an orthonormal panel: Ballard, Demmel, Grigori,
// Jacquelin, Knight, Nguyen, Solomonik 2015), and H(0) ... H(31) = I - V T V^T with T = -U V_1^{-T} (V_1: V's top 32 rows).  So
// V, T, R are Householder's, to rounding, and the trailing columns and Q are
// formed with blocked products as before.
//
// Q1 departs from orthonormal by eps cond(P)^2; the second pass brings it to eps
// while that is well below 1.  A panel whose G1 has no Cholesky factor or whose
// |G2 - I| exceeds 1e-4 (columns dependent to about 1e-6) sets `bad`, and the
// caller factors the matrix anew column by column.  So does a column with (next to)
// nothing below its diagonal, |pivot| = 1 to rounding: dlarfg keeps its sign when
// the rest is exactly zero (tau = 0), which the products cannot tell.
//
// Measured, one panel of 65536 rows: 5 launches, 85 us in all (34 and 930 us);
// Q and R of the five factors of a 65536 x 16384 sketch with range 401 (X^T, Y,
// two 803 x 401, one 401 x 401): 28 -> 9.5 ms.
#include <algorithm>

#include "linalg.hpp"
#include "util.hpp"

namespace skema {
namespace {

constexpr int kNb = 32;       // panel columns
constexpr int kMulWaves = 16; // waves of a panel product's block
constexpr int kOne = 512;     // threads of the one-block kernels
constexpr int kPairs = 3;     // 16 x 16 tiles of a panel's Gram: (0,0), (0,1), (1,1)

__device__ __forceinline__ void wave_order() {  // LDS accesses of a wave complete in issue order
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ double read_lane(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l), hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}

// D = P M (mp x 32 times 32 x 32 upper triangular; the identity when M is
// null), stored over P from row `from` on (STORE), and the Gram of D's columns,
// summed per block into part (GRAM).  A wave takes 16 rows at a time.  P as the
// A operand (rows on lane % 16) and M as the B operand leave D with columns on
// lane % 16 and rows on lane / 16 + 4 v: the operand layout of D^T D for both
// sides, so the Gram needs no transpose.  Bound by reading (and writing) P: 16.8
// MB at 65536 rows.
template <bool GRAM, bool STORE>
__global__ __launch_bounds__(64 * kMulWaves) void k_panel_mul(double* P, int64_t lda, int64_t mp, int jb, const double* M,
                                                              int64_t from, double* part) {
  __shared__ double red[GRAM ? kMulWaves * kPairs * 64 : 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  double mf[12];  // M's columns 0..15 (rows 0..15; below is zero), then 16..31
#pragma unroll
  for (int s = 0; s < 12; ++s) {
    const int r = 4 * (s < 4 ? s : s - 4) + lq, c = (s < 4 ? 0 : 16) + l16;
    mf[s] = M ? M[r * kNb + c] : (r == c ? 1.0 : 0.0);
  }
  d4 gr[kPairs];
#pragma unroll
  for (int q = 0; q < kPairs; ++q) gr[q] = d4{0.0, 0.0, 0.0, 0.0};
  const int tiles = (int)((mp + 15) / 16), stride = gridDim.x * kMulWaves;
  // byte offsets of the operand's columns 4 s + lq and of the result's 16 y + l16
  uint32_t oc[8], od[2];
#pragma unroll
  for (int s = 0; s < 8; ++s) oc[s] = (uint32_t)(4 * s + lq < jb ? 4 * s + lq : jb - 1) * (uint32_t)lda * 8u;
#pragma unroll
  for (int y = 0; y < 2; ++y) od[y] = ((uint32_t)(16 * y + l16) * (uint32_t)lda + (uint32_t)lq) * 8u;
  auto load = [&](int t, double (&x)[8]) {  // rows past the end: zero
    const char* base = reinterpret_cast<const char*>(P + 16 * (int64_t)t);
    const int left = (int)(mp - 16 * (int64_t)t - 1 < 15 ? mp - 16 * (int64_t)t - 1 : 15);
    const uint32_t orow = 8u * (uint32_t)(l16 < left ? l16 : left);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const double v = *reinterpret_cast<const double*>(base + (oc[s] + orow));
      x[s] = l16 <= left && 4 * s + lq < jb ? v : 0.0;
    }
  };
  double x[8], nx[8];
  int t = blockIdx.x * kMulWaves + wave;
  if (t < tiles) load(t, x);
  for (; t < tiles; t += stride) {
    load(t + stride < tiles ? t + stride : t, nx);
    d4 d[2];
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      d[y] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 4 * (y + 1); ++s)
        d[y] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[s], mf[4 * y + s], d[y], 0, 0, 0);
    }
    if (GRAM) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        gr[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(d[0][v], d[0][v], gr[0], 0, 0, 0);
        gr[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(d[0][v], d[1][v], gr[1], 0, 0, 0);
        gr[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(d[1][v], d[1][v], gr[2], 0, 0, 0);
      }
    }
    if (STORE) {
      char* base = reinterpret_cast<char*>(P + 16 * (int64_t)t);
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int64_t row = 16 * (int64_t)t + lq + 4 * v;
          if (row >= from && row < mp && 16 * y + l16 < jb)
            *reinterpret_cast<double*>(base + (od[y] + 32u * (uint32_t)v)) = d[y][v];
        }
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) x[s] = nx[s];
  }
  if (GRAM) {
    // one of the four result registers at a time, to keep the buffer small
#pragma unroll
    for (int v = 0; v < 4; ++v) {
#pragma unroll
      for (int q = 0; q < kPairs; ++q) red[(wave * kPairs + q) * 64 + lane] = gr[q][v];
      __syncthreads();
      if (tid < kPairs * 64) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kMulWaves; ++w) s += red[w * kPairs * 64 + tid];
        part[((int64_t)blockIdx.x * 4 + v) * (kPairs * 64) + tid] = s;
      }
      __syncthreads();
    }
  }
}

// G (32 x 32, symmetric) from the blocks' partial Grams, in block order; the
// padding past jb columns is the identity.
__device__ __forceinline__ void gather_gram(const double* part, int nblk, int jb, double (*G)[kNb + 1]) {
  constexpr int PER = 4 * kPairs * 64;
  for (int e = threadIdx.x; e < PER; e += kOne) {
    double s = 0.0;
#pragma unroll 32
    for (int b = 0; b < nblk; ++b) s += part[(int64_t)b * PER + e];
    const int v = e / (kPairs * 64), q = e / 64 % kPairs, l = e % 64;
    const int i = (q == 2 ? 16 : 0) + l / 16 + 4 * v, j = (q == 0 ? 0 : 16) + l % 16;
    const bool pad = i >= jb || j >= jb;
    s = pad ? (i == j ? 1.0 : 0.0) : s;
    G[i][j] = s;
    if (q == 1) G[j][i] = s;
  }
  __syncthreads();
}

// Lower Cholesky factor L of G (L L^T = G) and X = L^{-T}, by one wave: lane i
// < 32 forms row i of L, lane 32 + i row i of X, which obey the same recurrence
// over the rows of L (L_ij = (G_ij - sum_t L_it L_jt) / L_jj, X_ij = (I_ij -
// sum_t X_it L_jt) / L_jj, t < j).  Row j's entries come from LDS a step early,
// the last of them straight from lane j.  False when a pivot is not positive.
__device__ bool chol_and_inverse(const double (*G)[kNb + 1], double (*L)[kNb + 1], double (*X)[kNb + 1]) {
  const int lane = threadIdx.x & 63, i = lane & 31;
  const bool inv = lane >= 32;
  double (*out)[kNb + 1] = inv ? X : L;
  double h[kNb];
  double cur[kNb], nxt[kNb];
  bool ok = true;
#pragma unroll
  for (int j = 0; j < kNb; ++j) {
    if (j + 1 < kNb) {
#pragma unroll
      for (int t = 0; t < j; ++t) nxt[t] = L[j + 1][t];
    }
    double v = inv ? (i == j ? 1.0 : 0.0) : G[i][j];
    double w = 0.0;
#pragma unroll
    for (int t = 0; t + 1 < j; ++t) {
      if (t & 1) w -= h[t] * cur[t];
      else v -= h[t] * cur[t];
    }
    v += w;
    if (j > 0) v -= h[j - 1] * read_lane(h[j - 1], j);
    const double d = read_lane(v, j);
    ok = ok && d > 0.0;
    // 1 / sqrt(d) to rounding
    double y = __builtin_amdgcn_rsq(d);
    y = y * (1.5 - 0.5 * d * y * y);
    y = y * (1.5 - 0.5 * d * y * y);
    h[j] = inv || i >= j ? v * y : 0.0;
    out[i][j] = h[j];
    wave_order();
#pragma unroll
    for (int t = 0; t < j; ++t) cur[t] = nxt[t];
  }
  return ok;
}

// After G1: R1 (as its transpose L) and R1^{-1}.
__global__ __launch_bounds__(kOne) void k_panel_chol(const double* part, int nblk, int jb, double* R1, double* Minv,
                                                     int* bad) {
  __shared__ double G[kNb][kNb + 1], L[kNb][kNb + 1], X[kNb][kNb + 1];
  __shared__ int good;
  gather_gram(part, nblk, jb, G);
  if (threadIdx.x < 64) {
    const bool ok = chol_and_inverse(G, L, X);
    if (threadIdx.x == 0) good = ok;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kNb * kNb; e += kOne) {
    const int i = e / kNb, j = e % kNb;
    R1[e] = good ? (i <= j ? L[j][i] : 0.0) : (i == j ? 1.0 : 0.0);
    Minv[e] = good ? (i <= j ? X[i][j] : 0.0) : (i == j ? 1.0 : 0.0);
  }
  if (!good && threadIdx.x == 0) *bad = 1;
}

// After G2: the panel's R (diagonal block), T, V's top rows (written over P's)
// and M with V's other rows = Q1 M.  square: the panel has no row below its
// last column, whose reflector is then the identity (dlarfg of length 1).
__global__ __launch_bounds__(kOne) void k_panel_reflect(const double* part, int nblk, int jb, int square, double* P,
                                                        int64_t lda, const double* R1, double* Mout, double* Rd, double* T,
                                                        int* bad) {
  __shared__ double G[kNb][kNb + 1], L[kNb][kNb + 1], X[kNb][kNb + 1], A[kNb][kNb + 1], B[kNb][kNb + 1];
  __shared__ double U[kNb][kNb + 1], V[kNb][kNb + 1], Ui[kNb][kNb + 1];
  __shared__ double D[kNb];
  __shared__ double wmax[kOne / 64];
  __shared__ int good;
  constexpr int NE = kNb * kNb / kOne;  // elements per thread: (i0 + q * kOne / kNb, j)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i0 = tid / kNb, j = tid % kNb;
  auto row = [&](int q) { return i0 + q * (kOne / kNb); };
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    const int i = row(q);
    A[i][j] = i < jb && j < jb ? P[i + (int64_t)j * lda] : 0.0;
    B[i][j] = R1[i * kNb + j];
  }
  gather_gram(part, nblk, jb, G);
  // |G2 - I|, NaN counting as infinite
  double e = 0.0;
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    const double v = fabs(G[row(q)][j] - (row(q) == j ? 1.0 : 0.0));
    e = fmax(e, v <= 1e300 ? v : 1e300);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) e = fmax(e, __shfl_xor(e, o));
  if (lane == 0) wmax[wave] = e;
  if (tid == 0) good = 1;
  __syncthreads();
  e = 0.0;
#pragma unroll
  for (int w = 0; w < kOne / 64; ++w) e = fmax(e, wmax[w]);
  // R2^T = L and R2^{-1} = X.  With E = G2 - I below 1e-9, R2 = I + (E's upper
  // triangle, diagonal halved) and its inverse I - the same, to E^2 < eps.
  if (e <= 1e-9) {
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const int i = row(q);
      const double u = i < j ? G[i][j] : (i == j ? 0.5 * (G[i][i] - 1.0) : 0.0);
      const double one = i == j ? 1.0 : 0.0;
      L[j][i] = one + u;
      X[i][j] = one - u;
    }
  } else if (e <= 1e-4) {
    if (tid < 64) {
      const bool ok = chol_and_inverse(G, L, X);
      if (tid == 0) good = ok;
    }
  } else if (tid == 0) {
    good = 0;
  }
  __syncthreads();
  if (!good) {
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const int i = row(q);
      Mout[i * kNb + j] = i == j ? 1.0 : 0.0;
      Rd[i * kNb + j] = T[i * kNb + j] = 0.0;
    }
    if (tid == 0) *bad = 1;
    return;
  }
  double r[NE], qt[NE];
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    const int i = row(q);
    r[q] = qt[q] = 0.0;
#pragma unroll
    for (int t = 0; t < kNb; ++t) {
      r[q] += t >= i && t <= j ? L[t][i] * B[t][j] : 0.0;  // R' = R2 R1
      qt[q] += t <= j ? A[i][t] * X[t][j] : 0.0;           // Q's top rows
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NE; ++q) A[row(q)][j] = qt[q];
  __syncthreads();
  // LU of Q D - I, lane i < 32 holding row i of what is left of Q's top rows;
  // lane 32 + i forms row i of U^{-1} (the same elimination from zero).
  if (tid < 64) {
    const int li = lane & 31;
    const bool inv = lane >= 32;
    double m[kNb];
#pragma unroll
    for (int c = 0; c < kNb; ++c) m[c] = inv ? 0.0 : A[li][c];
    double dj[kNb];
    bool alone = false;  // a column with nothing below its diagonal
#pragma unroll
    for (int c = 0; c < kNb; ++c) {
      const double piv = read_lane(m[c], c);
      const bool none = square && c == jb - 1;
      alone = alone || (c < jb && !none && fabs(piv) > 1.0 - 1e-13);
      const double d = none ? copysign(1.0, piv) : -copysign(1.0, piv);
      const double p = none ? 0.0 : d * piv - 1.0;
      const double rp = none ? 0.0 : 1.0 / p;
      dj[c] = d;
      double f;
      if (inv) f = (d * m[c] + (li == c ? 1.0 : 0.0)) * rp;
      else f = li > c ? d * m[c] * rp : 0.0;
      if (inv) Ui[li][c] = f;
      else {
        V[li][c] = li > c ? f : (li == c ? 1.0 : 0.0);
        U[li][c] = li < c ? d * m[c] : (li == c ? p : 0.0);
      }
#pragma unroll
      for (int t = c + 1; t < kNb; ++t) m[t] -= f * read_lane(m[t], c);
    }
    if (alone && lane == 0) *bad = 1;
    if (lane < kNb) {
      double dl = 0.0;
#pragma unroll
      for (int c = 0; c < kNb; ++c)
        if (c == lane) dl = dj[c];
      D[lane] = dl;
    }
  }
  __syncthreads();
  if (tid < 64) {
    // T V_1^T = -U, lane i row i of T (both halves alike)
    const int li = lane & 31;
    double t[kNb];
#pragma unroll
    for (int c = 0; c < kNb; ++c) {
      double v = -U[li][c], w = 0.0;
#pragma unroll
      for (int l = 0; l < c; ++l) {
        if (l & 1) w -= t[l] * V[c][l];
        else v -= t[l] * V[c][l];
      }
      t[c] = v + w;
    }
    if (lane < kNb) {
#pragma unroll
      for (int c = 0; c < kNb; ++c) T[c * kNb + li] = t[c];  // column-major
    }
  }
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    const int i = row(q);
    double s = 0.0;
#pragma unroll
    for (int l = 0; l < kNb; ++l) s += l >= i && l <= j ? X[i][l] * D[l] * Ui[l][j] : 0.0;
    Mout[i * kNb + j] = s;
    Rd[i * kNb + j] = i <= j ? D[i] * r[q] : 0.0;
    if (i < jb && j < jb) P[i + (int64_t)j * lda] = V[i][j];
  }
}

__global__ void k_thin_r(int64_t n, const double* A, int64_t lda, const double* Rd, double* R, int64_t ldr) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n * n) return;
  const int64_t i = e % n, c = e / n;
  double v = 0.0;
  if (i / kNb == c / kNb) v = Rd[(i / kNb) * kNb * kNb + (i % kNb) * kNb + c % kNb];
  else if (i < c) v = A[i + c * lda];
  R[i + c * ldr] = v;
}

__global__ void k_eye(int64_t rows, int64_t cols, double* Q, int64_t ldq) {
  for (int64_t c = blockIdx.y; c < cols; c += gridDim.y)
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < rows; i += (int64_t)gridDim.x * blockDim.x)
      Q[i + c * ldq] = i == c ? 1.0 : 0.0;
}

int mul_blocks(int64_t mp) { return (int)std::min<int64_t>(64, cdiv(cdiv(mp, 16), kMulWaves)); }

}  // namespace

bool thin_qr_products(hipStream_t st, int64_t m, int64_t n, double* A, int64_t lda, double* Q, int64_t ldq, double* R,
                      int64_t ldr, DevBuf* work, GemmWorkspace* gws) {
  SKEMA_REQUIRE(m >= n && n > 0 && lda >= m && ldq >= m, kErrShape, "thin_qr_products: bad shape");
  if (lda > (int64_t)1 << 23) return false;  // 32-bit byte offsets within a panel's 32 columns
  const int64_t np = cdiv(n, kNb), sq = kNb * kNb;
  // workspace: T and R's diagonal block of every panel, R1, the two
  // multipliers, two 32 x n products, the partial Grams, the flag
  const int64_t per = 4 * kPairs * 64;
  size_t o = 0;
  auto take = [&](int64_t count) {
    const size_t at = o;
    o += align_up((size_t)count * sizeof(double), 256);
    return at;
  };
  const size_t oT = take(np * sq), oRd = take(np * sq), oR1 = take(sq), oM1 = take(sq), oM2 = take(sq),
               oW1 = take(kNb * n), oW2 = take(kNb * n), oP = take(mul_blocks(m) * per), oF = take(1);
  work->reserve(o);
  char* b = work->as<char>();
  auto at = [&](size_t off) { return reinterpret_cast<double*>(b + off); };
  double *Tall = at(oT), *Rd = at(oRd), *R1 = at(oR1), *M1 = at(oM1), *M2 = at(oM2), *W1 = at(oW1), *W2 = at(oW2),
         *part = at(oP);
  int* bad = reinterpret_cast<int*>(b + oF);
  fill_i32(st, bad, 1, 0);
  const dim3 mulb(64 * kMulWaves);
  for (int64_t j0 = 0; j0 < n; j0 += kNb) {
    const int64_t jb = std::min<int64_t>(kNb, n - j0), mp = m - j0, n2 = n - j0 - jb, p = j0 / kNb;
    double* P = A + j0 + j0 * lda;
    const int nblk = mul_blocks(mp);
    hipLaunchKernelGGL((k_panel_mul<true, false>), dim3(nblk), mulb, 0, st, P, lda, mp, (int)jb, nullptr, (int64_t)0,
                       part);
    hipLaunchKernelGGL(k_panel_chol, dim3(1), dim3(kOne), 0, st, part, nblk, (int)jb, R1, M1, bad);
    hipLaunchKernelGGL((k_panel_mul<true, true>), dim3(nblk), mulb, 0, st, P, lda, mp, (int)jb, M1, (int64_t)0, part);
    hipLaunchKernelGGL(k_panel_reflect, dim3(1), dim3(kOne), 0, st, part, nblk, (int)jb, mp == jb ? 1 : 0, P, lda, R1,
                       M2, Rd + p * sq, Tall + p * sq, bad);
    if (mp > jb)
      hipLaunchKernelGGL((k_panel_mul<false, true>), dim3((unsigned)std::min<int64_t>(256, cdiv(cdiv(mp, 16), kMulWaves))),
                         mulb, 0, st, P, lda, mp, (int)jb, M2, jb, nullptr);
    check_launch("k_panel_*");
    if (n2 == 0) break;
    // A2 <- (I - V T V^T)^T A2 = A2 - V (T^T (V^T A2))
    double* A2 = A + j0 + (j0 + jb) * lda;
    gemm_f64(st, 'T', 'N', jb, n2, mp, 1.0, P, lda, A2, lda, 0.0, W1, jb, gws);
    gemm_f64(st, 'T', 'N', jb, n2, jb, 1.0, Tall + p * sq, kNb, W1, jb, 0.0, W2, jb, gws);
    gemm_f64(st, 'N', 'N', mp, n2, jb, -1.0, P, lda, W2, jb, 1.0, A2, lda, gws);
  }
  int failed = 0;
  SKEMA_HIP(hipMemcpyAsync(&failed, bad, sizeof(int), hipMemcpyDeviceToHost, st));
  SKEMA_HIP(hipStreamSynchronize(st));
  if (failed) return false;
  if (R) {
    hipLaunchKernelGGL(k_thin_r, dim3((unsigned)cdiv(n * n, 256)), dim3(256), 0, st, n, A, lda, Rd, R, ldr);
    check_launch("k_thin_r");
  }
  // Q = H(0) ... H(n-1) [I; 0], last panel first: panel p acts on rows >= j0
  // only, where the columns before j0 are still zero
  hipLaunchKernelGGL(k_eye, dim3((unsigned)std::min<int64_t>(cdiv(m, 256), 64), (unsigned)std::min<int64_t>(n, 65535)),
                     dim3(256), 0, st, m, n, Q, ldq);
  check_launch("k_eye");
  for (int64_t p = np - 1; p >= 0; --p) {
    const int64_t j0 = p * kNb, jb = std::min<int64_t>(kNb, n - j0), mp = m - j0, nq = n - j0;
    const double* V = A + j0 + j0 * lda;
    double* Q2 = Q + j0 + j0 * ldq;
    gemm_f64(st, 'T', 'N', jb, nq, mp, 1.0, V, lda, Q2, ldq, 0.0, W1, jb, gws);
    gemm_f64(st, 'N', 'N', jb, nq, jb, 1.0, Tall + p * sq, kNb, W1, jb, 0.0, W2, jb, gws);
    gemm_f64(st, 'N', 'N', mp, nq, jb, -1.0, V, lda, W2, jb, 1.0, Q2, ldq, gws);
  }
  return true;
}

}  // namespace skema
