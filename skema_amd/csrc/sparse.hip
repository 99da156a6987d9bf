// Sparse kernels of the sketch path (sparse-sign maps, CSR windows).
// Bandwidth-bound gathers: consecutive lanes own consecutive output rows of a
// column-major result, so stores and the dense-operand loads coalesce, and
// no two threads ever accumulate into the same element.
#include <algorithm>
#include <vector>

#include "sparse.hpp"
#include "util.hpp"

namespace skema {
namespace {

unsigned blocks_for(int64_t n, int bs = 256) {
  int64_t b = cdiv(n, bs);
  if (b > (int64_t)1 << 30) b = (int64_t)1 << 30;
  return (unsigned)(b < 1 ? 1 : b);
}

__device__ __forceinline__ int64_t lower_bound_col(const int32_t* ci, int64_t lo, int64_t hi, int64_t key) {
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (ci[mid] < key) lo = mid + 1; else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ void put(const GemmOut& o, int64_t i, int64_t p, double v) {
  if (p < o.nsplit) {
    double* c = o.C1 + i + p * o.ldc1;
    *c = (o.beta1 != 0.0) ? o.alpha1 * v + o.beta1 * *c : o.alpha1 * v;
  } else {
    double* c = o.C2 + i + (p - o.nsplit) * o.ldc2;
    *c = (o.beta2 != 0.0) ? o.alpha2 * v + o.beta2 * *c : o.alpha2 * v;
  }
}

__global__ void k_spmm_csr_rows(const int64_t* rp, const int32_t* ci, const double* cv, int64_t r0, int64_t R,
                                int64_t c0, int64_t c1, bool windowed, double alpha, const double* B, int64_t ldb,
                                int64_t N, double beta, double* C, int64_t ldc) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= R * N) return;
  const int64_t p = g % R, j = g / R;
  int64_t lo = rp[r0 + p], hi = rp[r0 + p + 1];
  if (windowed) {
    const int64_t a = lower_bound_col(ci, lo, hi, c0);
    hi = lower_bound_col(ci, a, hi, c1);
    lo = a;
  }
  const double* b = B + j * ldb - c0;
  double acc = 0.0;
  for (int64_t e = lo; e < hi; ++e) acc += cv[e] * b[ci[e]];
  double* c = C + p + j * ldc;
  *c = (beta != 0.0) ? alpha * acc + beta * *c : alpha * acc;
}

// Split form for short M and long rows of S: block (p, z) sums the z-th
// chunk of row p's nonzeros for all M rows of B (thread = row i), partials
// part[z][i + p M] reduced in a fixed order by k_spmm_split_reduce.  Bound by
// the latency of the gathered columns of B, so kSplitLoads of them are in
// flight at a time; the sum keeps the nonzeros' order.  M = 203, 160000 nonzeros
// in 203 rows: 56 -> 31 us.
constexpr int kSplitLoads = 8;
__global__ __launch_bounds__(256) void k_spmm_dense_csrT_split(int64_t M, const double* __restrict__ B, int64_t ldb,
                                                               const int64_t* __restrict__ rp,
                                                               const int32_t* __restrict__ ci,
                                                               const double* __restrict__ cv, int64_t R, int64_t chunk,
                                                               double* __restrict__ part) {
  const int64_t p = blockIdx.x, z = blockIdx.y;
  const int64_t lo = rp[p] + z * chunk, hi0 = rp[p + 1];
  const int64_t hi = (lo + chunk < hi0) ? lo + chunk : hi0;
  for (int64_t i = threadIdx.x; i < M; i += blockDim.x) {
    double acc = 0.0;
    int64_t e = lo;
    for (; e + kSplitLoads <= hi; e += kSplitLoads) {
      double b[kSplitLoads];
#pragma unroll
      for (int q = 0; q < kSplitLoads; ++q) b[q] = B[i + (int64_t)ci[e + q] * ldb];
#pragma unroll
      for (int q = 0; q < kSplitLoads; ++q) acc += cv[e + q] * b[q];
    }
    for (; e < hi; ++e) acc += cv[e] * B[i + (int64_t)ci[e] * ldb];
    part[z * M * R + i + p * M] = acc;
  }
}
__global__ void k_spmm_split_reduce(int64_t M, int64_t R, int splits, const double* part, GemmOut o) {
  const int64_t total = M * R;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    double v = 0.0;
    for (int z = 0; z < splits; ++z) v += part[(int64_t)z * total + e];
    put(o, e % M, e / M, v);
  }
}

__global__ void k_spmm_dense_csrT(int64_t M, const double* B, int64_t ldb, const int64_t* rp, const int32_t* ci,
                                  const double* cv, int64_t R, GemmOut o) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= M * R) return;
  const int64_t i = g % M, p = g / M;
  double acc = 0.0;
  for (int64_t e = rp[p]; e < rp[p + 1]; ++e) acc += cv[e] * B[i + (int64_t)ci[e] * ldb];
  put(o, i, p, acc);
}

// ---- CSR window -> CSC ----------------------------------------------------
__global__ void k_inspect_csr(const int64_t* rowptr, int64_t rows, const int32_t* col, int64_t cols, int64_t room,
                              int64_t* out) {
  const int64_t base = rowptr[0], end = rowptr[rows];
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
  if (i0 == 0) {
    out[0] = base;
    out[1] = end;
  }
  unsigned long long bad = 0;
  for (int64_t i = i0; i < rows; i += step)
    if (rowptr[i + 1] < rowptr[i]) bad |= 1;
  if (base >= 0 && end >= base && end <= room && end - base < ((int64_t)1 << 31))
    for (int64_t e = base + i0; e < end; e += step) {
      const int32_t c = col[e];
      if (c < 0 || c >= cols) bad |= 2;
    }
  if (bad) atomicOr(reinterpret_cast<unsigned long long*>(out + 2), bad);
}

__global__ void k_count_cols(const int64_t* rowptr, int64_t rows, const int32_t* col, int* counts) {
  const int64_t base = rowptr[0];
  const int64_t nnz = rowptr[rows] - base;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nnz; e += (int64_t)gridDim.x * blockDim.x)
    atomicAdd(&counts[col[base + e]], 1);
}

// Column counts per row block in LDS (cols <= kHistCols, the histogram sized
// to cols in dynamic LDS): block b takes rows [b R, (b+1) R), walks its
// nonzeros in storage order (coalesced), counts them per column in LDS and
// writes the histogram to T[b][0..cols).  No global atomics.
constexpr int kHistCols = 32768;
__global__ __launch_bounds__(1024) void k_count_cols_blocked(const int64_t* rowptr, int64_t rows, const int32_t* col,
                                                            int64_t cols, int64_t R, int* T) {
  extern __shared__ int hist[];
  const int64_t b = blockIdx.x;
  for (int64_t c = threadIdx.x; c < cols; c += 1024) hist[c] = 0;
  __syncthreads();
  const int64_t r0 = b * R, r1 = (r0 + R < rows) ? r0 + R : rows;
  if (r0 < r1) {
    const int64_t e1 = rowptr[r1];
    for (int64_t e = rowptr[r0] + threadIdx.x; e < e1; e += 1024) atomicAdd(&hist[col[e]], 1);
  }
  __syncthreads();
  for (int64_t c = threadIdx.x; c < cols; c += 1024) T[b * cols + c] = hist[c];
}
// Per column: T[b][c] <- sum_{b' < b} T[b'][c] (exclusive, in block order),
// counts[c] <- the column total.
// Sixteen row blocks' counts are loaded before any is overwritten, so the
// loads of a batch are in flight together.
__global__ void k_scan_blocks(int64_t nb, int64_t cols, int* T, int* counts) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= cols) return;
  constexpr int kB = 16;
  int run = 0;
  for (int64_t b0 = 0; b0 < nb; b0 += kB) {
    int t[kB];
#pragma unroll
    for (int j = 0; j < kB; ++j) t[j] = (b0 + j < nb) ? T[(b0 + j) * cols + c] : 0;
#pragma unroll
    for (int j = 0; j < kB; ++j) {
      if (b0 + j < nb) T[(b0 + j) * cols + c] = run;
      run += t[j];
    }
  }
  counts[c] = run;
}
// Scatter of block b's rows into its own sub-range of every column:
// cursor[c] = ptr[c] + T[b][c] in LDS, one LDS atomic per nonzero.  The
// block's nonzeros are walked in storage order (coalesced reads); the row of
// nonzero e is found by binary search in the block's slice of rowptr, which
// is staged in LDS after the cursors (R + 1 entries, relative to the slice
// start).
__global__ __launch_bounds__(1024) void k_fill_csc_blocked(const int64_t* rowptr, int64_t rows, const int32_t* col,
                                                          const double* val, int64_t cols, int64_t R, const int* T,
                                                          const int64_t* ptr, int32_t* orow, double* oval) {
  extern __shared__ int lds[];
  int* cur = lds;
  int* rp = lds + cols;  // rowptr[r0 .. r1] - rowptr[r0]
  const int64_t b = blockIdx.x;
  const int64_t r0 = b * R, r1 = (r0 + R < rows) ? r0 + R : rows;
  if (r0 >= r1) return;  // whole block: no barrier is skipped by part of it
  const int64_t e0 = rowptr[r0];
  const int nr = (int)(r1 - r0);
  for (int64_t c = threadIdx.x; c < cols; c += 1024) cur[c] = (int)ptr[c] + T[b * cols + c];
  for (int i = threadIdx.x; i <= nr; i += 1024) rp[i] = (int)(rowptr[r0 + i] - e0);
  __syncthreads();
  const int ne = rp[nr];
  for (int e = threadIdx.x; e < ne; e += 1024) {
    // last row start <= e
    int lo = 0, hi = nr - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (rp[mid] <= e) lo = mid; else hi = mid - 1;
    }
    const int32_t c = col[e0 + e];
    const int pos = atomicAdd(&cur[c], 1);
    orow[pos] = (int32_t)(r0 + lo);
    oval[pos] = val[e0 + e];
  }
}

// Exclusive scan of counts[0..n) into ptr[0..n] by one block of 1024 threads.
// Tiles of 8192 counts: coalesced loads into LDS, each thread sums its 8
// consecutive entries, a block scan of the 1024 sums, coalesced writes of the
// exclusive prefixes, and the tile total carried to the next tile.
__global__ __launch_bounds__(1024) void k_scan_counts(const int* counts, int64_t n, int64_t* ptr) {
  constexpr int kPer = 8, kTile = 1024 * kPer;
  __shared__ int64_t part[1024];
  __shared__ int64_t tile[kTile];
  const int t = threadIdx.x;
  int64_t carry = 0;
  for (int64_t t0 = 0; t0 < n; t0 += kTile) {
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int64_t i = t0 + j * 1024 + t;
      tile[j * 1024 + t] = i < n ? counts[i] : 0;
    }
    __syncthreads();
    int64_t s = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) s += tile[t * kPer + j];
    part[t] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
      const int64_t v = (t >= off) ? part[t - off] : 0;
      __syncthreads();
      part[t] += v;
      __syncthreads();
    }
    int64_t run = carry + part[t] - s;  // exclusive prefix of this thread's 8 entries
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int64_t c = tile[t * kPer + j];
      tile[t * kPer + j] = run;
      run += c;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int64_t i = t0 + j * 1024 + t;
      if (i < n) ptr[i] = tile[j * 1024 + t];
    }
    carry += part[1023];
    __syncthreads();
  }
  if (t == 0) ptr[n] = carry;
}

__global__ void k_fill_csc(const int64_t* rowptr, int64_t rows, const int32_t* col, const double* val, int* cursor,
                           const int64_t* ptr, int32_t* orow, double* oval) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows) return;
  for (int64_t e = rowptr[i]; e < rowptr[i + 1]; ++e) {
    const int32_t c = col[e];
    const int64_t pos = ptr[c] + atomicAdd(&cursor[c], 1);
    orow[pos] = (int32_t)i;
    oval[pos] = val[e];
  }
}

// Sort of each column segment by (row, value): makes the order of summation
// independent of the atomic placement above.  One 64-thread block per column:
// a bitonic sort in LDS for up to 1024 entries, insertion sort by one thread
// above that.
constexpr int kSortMax = 1024;
__global__ __launch_bounds__(64) void k_sort_columns(const int64_t* ptr, int32_t* row, double* val) {
  __shared__ int32_t kr[kSortMax];
  __shared__ double kv[kSortMax];
  const int tid = threadIdx.x;
  const int64_t c = blockIdx.x;
  const int64_t lo = ptr[c], hi = ptr[c + 1], len = hi - lo;
  if (len <= 1) return;
  if (len > kSortMax) {
    if (tid != 0) return;
    for (int64_t a = lo + 1; a < hi; ++a) {
      const int32_t r = row[a];
      const double v = val[a];
      int64_t b = a - 1;
      while (b >= lo && (row[b] > r || (row[b] == r && val[b] > v))) {
        row[b + 1] = row[b];
        val[b + 1] = val[b];
        --b;
      }
      row[b + 1] = r;
      val[b + 1] = v;
    }
    return;
  }
  int n = 1;
  while (n < len) n <<= 1;
  for (int t = tid; t < n; t += 64) {
    const bool in = t < len;
    kr[t] = in ? row[lo + t] : INT32_MAX;
    kv[t] = in ? val[lo + t] : INFINITY;
  }
  __syncthreads();
  for (int k = 2; k <= n; k <<= 1)
    for (int jj = k >> 1; jj > 0; jj >>= 1) {
      for (int t = tid; t < n; t += 64) {
        const int u = t ^ jj;
        if (u > t) {
          const bool up = (t & k) == 0;
          const bool gt = kr[t] > kr[u] || (kr[t] == kr[u] && kv[t] > kv[u]);
          if (gt == up) {
            const int32_t r = kr[t];
            kr[t] = kr[u];
            kr[u] = r;
            const double v = kv[t];
            kv[t] = kv[u];
            kv[u] = v;
          }
        }
      }
      __syncthreads();
    }
  for (int t = tid; t < len; t += 64) {
    row[lo + t] = kr[t];
    val[lo + t] = kv[t];
  }
}

// X(p, j) = nu X + eta sum over column j's entries (i, a) of a M(p, row0 + i): one
// wave per column and 64 PR rows p, the entries in order, four of them (and their
// map columns) in flight at a time.  With cw, a is weighted by cw[i / window].
template <int PR, bool CW>
__global__ __launch_bounds__(256) void k_csc_left_dense(const int64_t* __restrict__ ptr, const int32_t* __restrict__ row,
                                                        const double* __restrict__ val, int64_t cols,
                                                        const double* __restrict__ M, int64_t ldm, int64_t row0,
                                                        int64_t k, const double* __restrict__ cw, uint32_t window,
                                                        double eta, double nu, double* __restrict__ X, int64_t ldx) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t j = (int64_t)blockIdx.x * 4 + wave, p0 = (int64_t)blockIdx.y * (64 * PR);
  if (j >= cols) return;
  const int64_t lo = ptr[j], hi = ptr[j + 1];
  int64_t at[PR];  // this lane's rows (past k: the last one's, not stored)
#pragma unroll
  for (int r = 0; r < PR; ++r) at[r] = p0 + lane + 64 * r < k ? p0 + lane + 64 * r : k - 1;
  double acc[PR];
#pragma unroll
  for (int r = 0; r < PR; ++r) acc[r] = 0.0;
  auto term = [&](int64_t e, const double*& m) {
    const int32_t i = row[e];
    m = M + (row0 + i) * ldm;
    return CW ? val[e] * cw[(uint32_t)i / window] : val[e];
  };
  int64_t e = lo;
  for (; e + 4 <= hi; e += 4) {
    const double* m[4];
    double a[4], v[4][PR];
#pragma unroll
    for (int q = 0; q < 4; ++q) a[q] = term(e + q, m[q]);
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < PR; ++r) v[q][r] = m[q][at[r]];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < PR; ++r) acc[r] += a[q] * v[q][r];
  }
  for (; e < hi; ++e) {
    const double* m;
    const double a = term(e, m);
#pragma unroll
    for (int r = 0; r < PR; ++r) acc[r] += a * m[at[r]];
  }
#pragma unroll
  for (int r = 0; r < PR; ++r) {
    const int64_t p = p0 + lane + 64 * r;
    if (p < k) {
      double* x = X + p + j * ldx;
      *x = (nu != 0.0) ? nu * *x + eta * acc[r] : eta * acc[r];
    }
  }
}

__global__ void k_csc_left_sparse(const int64_t* ptr, const int32_t* row, const double* val, int64_t cols,
                                  const int64_t* mrp, const int32_t* mci, const double* mv, int64_t row0, int64_t k,
                                  double eta, double nu, double* X, int64_t ldx) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= cols) return;
  double* x = X + j * ldx;
  if (nu != 1.0)
    for (int64_t p = 0; p < k; ++p) x[p] = (nu != 0.0) ? nu * x[p] : 0.0;
  for (int64_t e = ptr[j]; e < ptr[j + 1]; ++e) {
    const double a = eta * val[e];
    const int64_t c = row0 + row[e];
    for (int64_t f = mrp[c]; f < mrp[c + 1]; ++f) x[mci[f]] += a * mv[f];
  }
}

// out(i, p) = sum over row i's entries (j, a) of a M(p, j): RT rows and LP PR
// map rows p a block.  A row is taken by LP lanes of a wave (16 or 32 where there
// are no more map rows, so that a wave has four or two rows at once), a wave's
// rows one after another (entries in order, four and their map columns in flight),
// then through LDS so that a column of the output is written RT rows at a time
// (16: 128 bytes).  One thread per output with p fastest wrote every 8 bytes to a
// line of its own: 4096 x 304 outputs with 15 entries a row took 48 us, 24 here.
template <int PR, int RT, int LP>
__global__ __launch_bounds__(256) void k_csr_right_dense(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                                         const double* __restrict__ val, int64_t rows,
                                                         const double* __restrict__ M, int64_t ldm, int64_t kk, GemmOut o) {
  constexpr int AT = 256 / LP;  // rows at a time
  static_assert(RT % AT == 0, "whole passes");
  __shared__ double tile[LP * PR][RT + 1];
  const int tid = threadIdx.x, lane = tid % LP;
  const int own = LP == 64 ? __builtin_amdgcn_readfirstlane(tid / 64) : tid / LP;
  const int64_t r0 = (int64_t)blockIdx.x * RT, p0 = (int64_t)blockIdx.y * (LP * PR);
  int64_t at[PR];
#pragma unroll
  for (int r = 0; r < PR; ++r) at[r] = p0 + lane + LP * r < kk ? p0 + lane + LP * r : kk - 1;
  for (int q = 0; q < RT / AT; ++q) {
    const int64_t i = r0 + AT * q + own;
    if (i >= rows) break;
    const int64_t lo = rowptr[i], hi = rowptr[i + 1];
    double acc[PR];
#pragma unroll
    for (int r = 0; r < PR; ++r) acc[r] = 0.0;
    int64_t e = lo;
    for (; e + 4 <= hi; e += 4) {
      const double* m[4];
      double a[4], v[4][PR];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        a[t] = val[e + t];
        m[t] = M + (int64_t)col[e + t] * ldm;
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < PR; ++r) v[t][r] = m[t][at[r]];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < PR; ++r) acc[r] += a[t] * v[t][r];
    }
    for (; e < hi; ++e) {
      const double a = val[e];
      const double* m = M + (int64_t)col[e] * ldm;
#pragma unroll
      for (int r = 0; r < PR; ++r) acc[r] += a * m[at[r]];
    }
#pragma unroll
    for (int r = 0; r < PR; ++r) tile[lane + LP * r][AT * q + own] = acc[r];
  }
  __syncthreads();
  for (int x = tid; x < LP * PR * RT; x += 256) {
    const int ii = x % RT, pp = x / RT;
    if (r0 + ii < rows && p0 + pp < kk) put(o, r0 + ii, p0 + pp, tile[pp][ii]);
  }
}

__global__ void k_csr_right_sparse(const int64_t* rowptr, const int32_t* col, const double* val, int64_t rows,
                                   const int64_t* mrp, const int32_t* mci, const double* mv, int64_t kk, GemmOut o) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows) return;
  // beta pass
  for (int64_t p = 0; p < kk; ++p) {
    if (p < o.nsplit) {
      double* c = o.C1 + i + p * o.ldc1;
      *c = (o.beta1 != 0.0) ? o.beta1 * *c : 0.0;
    } else {
      double* c = o.C2 + i + (p - o.nsplit) * o.ldc2;
      *c = (o.beta2 != 0.0) ? o.beta2 * *c : 0.0;
    }
  }
  for (int64_t e = rowptr[i]; e < rowptr[i + 1]; ++e) {
    const double a = val[e];
    const int32_t j = col[e];
    for (int64_t f = mrp[j]; f < mrp[j + 1]; ++f) {
      const int64_t p = mci[f];
      if (p < o.nsplit) o.C1[i + p * o.ldc1] += o.alpha1 * (a * mv[f]);
      else o.C2[i + (p - o.nsplit) * o.ldc2] += o.alpha2 * (a * mv[f]);
    }
  }
}

}  // namespace

void spmm_csr_rows(hipStream_t st, const Csr& S, int64_t r0, int64_t r1, int64_t c0, int64_t c1, double alpha,
                   const double* B, int64_t ldb, int64_t N, double beta, double* C, int64_t ldc) {
  const int64_t R = r1 - r0;
  SKEMA_REQUIRE(r0 >= 0 && r1 <= S.rows && R >= 0 && c0 >= 0 && c1 <= S.cols && c0 <= c1, kErrShape,
                "spmm_csr_rows: range outside the map");
  if (R == 0 || N == 0) return;
  const bool windowed = !(c0 == 0 && c1 == S.cols);
  hipLaunchKernelGGL(k_spmm_csr_rows, dim3(blocks_for(R * N)), dim3(256), 0, st, S.rp(), S.ci(), S.v(), r0, R, c0,
                     c1, windowed, alpha, B, ldb, N, beta, C, ldc);
  check_launch("k_spmm_csr_rows");
}

void spmm_dense_csrT(hipStream_t st, int64_t M, const double* B, int64_t ldb, const Csr& S, const GemmOut& out,
                     DevBuf* ws) {
  if (M == 0 || S.rows == 0) return;
  // few output elements and long rows of S: split each row's nonzeros so the
  // grid covers the chip (partials then a fixed-order sum)
  const int64_t avg = S.nnz / S.rows;
  if (ws && M <= 1024 && M * S.rows < 256 * 1024 && avg >= 64) {
    const int64_t splits = std::min<int64_t>(64, std::max<int64_t>(1, avg / 32));
    // the longest row bounds the chunk (read once per CSR and kept)
    if (S.max_row < 0) {
      std::vector<int64_t> h((size_t)S.rows + 1);
      SKEMA_HIP(hipMemcpyAsync(h.data(), S.rp(), h.size() * sizeof(int64_t), hipMemcpyDeviceToHost, st));
      SKEMA_HIP(hipStreamSynchronize(st));
      int64_t mr = 0;
      for (int64_t r = 0; r < S.rows; ++r) mr = std::max(mr, h[(size_t)r + 1] - h[(size_t)r]);
      S.max_row = mr;
    }
    const int64_t maxrow = S.max_row;
    const int64_t chunk = std::max<int64_t>(1, cdiv(maxrow, splits));
    const int64_t zs = cdiv(maxrow, chunk);
    ws->reserve((size_t)zs * M * S.rows * sizeof(double));
    double* part = ws->as<double>();
    const unsigned threads = (unsigned)std::min<int64_t>(256, cdiv(M, 64) * 64);
    hipLaunchKernelGGL(k_spmm_dense_csrT_split, dim3((unsigned)S.rows, (unsigned)zs), dim3(threads), 0, st, M, B, ldb,
                       S.rp(), S.ci(), S.v(), S.rows, chunk, part);
    check_launch("k_spmm_dense_csrT_split");
    const unsigned nb = (unsigned)std::min<int64_t>(cdiv(M * S.rows, 256), 4096);
    hipLaunchKernelGGL(k_spmm_split_reduce, dim3(nb), dim3(256), 0, st, M, S.rows, (int)zs, part, out);
    check_launch("k_spmm_split_reduce");
    return;
  }
  hipLaunchKernelGGL(k_spmm_dense_csrT, dim3(blocks_for(M * S.rows)), dim3(256), 0, st, M, B, ldb, S.rp(), S.ci(),
                     S.v(), S.rows, out);
  check_launch("k_spmm_dense_csrT");
}

CsrInfo inspect_csr(Ctx* c, const int64_t* rowptr, const int32_t* col, int64_t rows, int64_t cols, int64_t room) {
  hipStream_t st = c->stream;
  constexpr size_t kBytes = 3 * sizeof(int64_t);
  if (!c->csr_dev.p) {
    c->csr_dev.alloc(kBytes);
    fill_i32(st, c->csr_dev.as<int>(), kBytes / sizeof(int), 0);
  }
  if (!c->csr_host.p) SKEMA_HIP(hipHostMalloc(&c->csr_host.p, kBytes, hipHostMallocDefault));
  int64_t* dev = c->csr_dev.as<int64_t>();
  const int64_t work = std::max(rows, room);
  const unsigned nb = (unsigned)std::max<int64_t>(1, std::min<int64_t>(cdiv(work, 256), 2048));
  hipLaunchKernelGGL(k_inspect_csr, dim3(nb), dim3(256), 0, st, rowptr, rows, col, cols, room, dev);
  check_launch("k_inspect_csr");
  SKEMA_HIP(hipMemcpyAsync(c->csr_host.p, dev, kBytes, hipMemcpyDeviceToHost, st));
  SKEMA_HIP(hipStreamSynchronize(st));
  const int64_t* h = static_cast<const int64_t*>(c->csr_host.p);
  const CsrInfo info{h[0], h[1], h[2]};
  if (info.flags) {
    // The caller refuses the window, so nothing after this waits for the clearing,
    // and the context's next inspection may run on another stream.
    fill_i32(st, reinterpret_cast<int*>(dev + 2), 2, 0);
    SKEMA_HIP(hipStreamSynchronize(st));
  }
  return info;
}

CscWindow csr_window_to_csc(hipStream_t st, const int64_t* rowptr, const int32_t* col, const double* val,
                            int64_t rows, int64_t cols, int64_t nnz, DevBuf& scratch, bool sorted) {
  const size_t o_cnt = 0;
  const size_t o_ptr = align_up((size_t)cols * sizeof(int) * 2, 256);
  const size_t o_row = o_ptr + align_up((size_t)(cols + 1) * sizeof(int64_t), 256);
  const size_t o_val = o_row + align_up((size_t)nnz * sizeof(int32_t), 256);
  // Row-blocked counts and placement in LDS when the columns fit (no global
  // atomics; one block per about 2048 nonzeros, 16 to 512 of them: the scan of
  // the blocks' counts reads cols ints a block, 35 us for 512 blocks of 3001
  // columns, 4 us for the 30 that 61000 nonzeros take); global atomic counters
  // otherwise.
  const int64_t nbk = std::max<int64_t>(16, std::min<int64_t>(512, cdiv(nnz, (int64_t)2048))), R = cdiv(rows, nbk);
  // (the fill keeps cols cursors and the R + 1 row starts of its slice in LDS)
  const bool blocked =
      cols <= kHistCols && rows >= 256 && nnz > 0 && (size_t)(cols + R + 1) * sizeof(int) <= 160 * 1024;
  const size_t o_T = o_val + align_up((size_t)nnz * sizeof(double), 256);
  const size_t total = o_T + (blocked ? align_up((size_t)nbk * cols * sizeof(int), 256) : 0);
  scratch.reserve(total);
  char* base = scratch.as<char>();
  int* counts = reinterpret_cast<int*>(base + o_cnt);
  int* cursor = counts + cols;
  CscWindow w;
  w.rows = rows;
  w.cols = cols;
  w.nnz = nnz;
  w.ptr = reinterpret_cast<int64_t*>(base + o_ptr);
  w.row = reinterpret_cast<int32_t*>(base + o_row);
  w.val = reinterpret_cast<double*>(base + o_val);
  int* T = blocked ? reinterpret_cast<int*>(base + o_T) : nullptr;
  if (blocked) {
    hipLaunchKernelGGL(k_count_cols_blocked, dim3((unsigned)nbk), dim3(1024), (size_t)cols * sizeof(int), st, rowptr,
                       rows, col, cols, R, T);
    hipLaunchKernelGGL(k_scan_blocks, dim3(blocks_for(cols)), dim3(256), 0, st, nbk, cols, T, counts);
  } else {
    fill_i32(st, counts, 2 * cols, 0);
    if (nnz > 0) {
      const unsigned nb = blocks_for(nnz) > 65536 ? 65536 : blocks_for(nnz);
      hipLaunchKernelGGL(k_count_cols, dim3(nb), dim3(256), 0, st, rowptr, rows, col, counts);
    }
  }
  hipLaunchKernelGGL(k_scan_counts, dim3(1), dim3(1024), 0, st, counts, cols, w.ptr);
  if (nnz > 0) {
    if (blocked)
      hipLaunchKernelGGL(k_fill_csc_blocked, dim3((unsigned)nbk), dim3(1024), (size_t)(cols + R + 1) * sizeof(int), st,
                         rowptr, rows, col, val, cols, R, T, w.ptr, w.row, w.val);
    else
      hipLaunchKernelGGL(k_fill_csc, dim3(blocks_for(rows)), dim3(256), 0, st, rowptr, rows, col, val, cursor, w.ptr,
                         w.row, w.val);
    if (sorted) hipLaunchKernelGGL(k_sort_columns, dim3((unsigned)cols), dim3(64), 0, st, w.ptr, w.row, w.val);
  }
  check_launch("csr_window_to_csc");
  return w;
}

void csc_left_dense(hipStream_t st, const CscWindow& H, const double* M, int64_t ldm, int64_t row0, int64_t k,
                    double eta, double nu, double* X, int64_t ldx, const double* cw, int64_t window) {
  if (k == 0 || H.cols == 0) return;
  const int pr = k <= 128 ? 2 : k <= 256 ? 4 : 8;  // map rows per lane
  const dim3 grid(blocks_for(H.cols, 4), (unsigned)cdiv(k, (int64_t)64 * pr));
#define SKEMA_LEFT(PR, CW)                                                                                            \
  hipLaunchKernelGGL((k_csc_left_dense<PR, CW>), grid, dim3(256), 0, st, H.ptr, H.row, H.val, H.cols, M, ldm, row0, k, \
                     cw, (uint32_t)window, eta, nu, X, ldx)
  if (cw) {
    if (pr == 2) SKEMA_LEFT(2, true);
    else if (pr == 4) SKEMA_LEFT(4, true);
    else SKEMA_LEFT(8, true);
  } else {
    if (pr == 2) SKEMA_LEFT(2, false);
    else if (pr == 4) SKEMA_LEFT(4, false);
    else SKEMA_LEFT(8, false);
  }
#undef SKEMA_LEFT
  check_launch("k_csc_left_dense");
}

void csc_left_sparse(hipStream_t st, const CscWindow& H, const Csr& Mt, int64_t row0, int64_t k, double eta,
                     double nu, double* X, int64_t ldx) {
  if (k == 0 || H.cols == 0) return;
  hipLaunchKernelGGL(k_csc_left_sparse, dim3(blocks_for(H.cols)), dim3(256), 0, st, H.ptr, H.row, H.val, H.cols,
                     Mt.rp(), Mt.ci(), Mt.v(), row0, k, eta, nu, X, ldx);
  check_launch("k_csc_left_sparse");
}

void csr_right_dense(hipStream_t st, const int64_t* rowptr, const int32_t* col, const double* val, int64_t rows,
                     const double* M, int64_t ldm, int64_t kk, const GemmOut& out) {
  if (rows == 0 || kk == 0) return;
  // Map rows in equal parts of at most 320 (five a lane: 44 KB of LDS, three blocks a
  // CU; 328 rows as 3 + 3 lots of 64, not 5 + 1), unless that leaves CUs without a
  // block: then 64 a block, and 4 rows a block instead of 16 where it still does.
  // Whole calls on windows with 300 entries a row, always 16 rows and all parts a
  // block -> so (one thread per output): 64 rows, 197 map rows 226 -> 73 us (143);
  // 1000 rows, 304 map rows 264 -> 200 (226).  Up to 32 map rows, a wave a row ->
  // several rows a wave: 60000 rows of 50, 9 map rows 148 -> 102 us (139).
  const int64_t parts = cdiv(kk, (int64_t)320), tall = cdiv(rows, (int64_t)16);
  int pr = (int)cdiv(cdiv(kk, (int64_t)64), parts);
  if (tall * parts < 256) pr = 1;
  const int64_t ny = cdiv(kk, (int64_t)64 * pr);
  const bool few = tall * ny < 256;
#define SKEMA_RIGHT(PR, RT, LP)                                                                                   \
  hipLaunchKernelGGL((k_csr_right_dense<PR, RT, LP>), dim3(blocks_for(rows, RT), (unsigned)ny), dim3(256), 0, st, \
                     rowptr, col, val, rows, M, ldm, kk, out)
  if (kk <= 16) SKEMA_RIGHT(1, 16, 16);
  else if (kk <= 32 && few) SKEMA_RIGHT(1, 8, 32);
  else if (kk <= 32) SKEMA_RIGHT(1, 16, 32);
  else if (few) SKEMA_RIGHT(1, 4, 64);
  else if (pr == 1) SKEMA_RIGHT(1, 16, 64);
  else if (pr == 2) SKEMA_RIGHT(2, 16, 64);
  else if (pr == 3) SKEMA_RIGHT(3, 16, 64);
  else if (pr == 4) SKEMA_RIGHT(4, 16, 64);
  else SKEMA_RIGHT(5, 16, 64);
#undef SKEMA_RIGHT
  check_launch("k_csr_right_dense");
}

void csr_right_sparse(hipStream_t st, const int64_t* rowptr, const int32_t* col, const double* val, int64_t rows,
                      const Csr& Mt, int64_t kk, const GemmOut& out) {
  if (rows == 0 || kk == 0) return;
  hipLaunchKernelGGL(k_csr_right_sparse, dim3(blocks_for(rows)), dim3(256), 0, st, rowptr, col, val, rows, Mt.rp(),
                     Mt.ci(), Mt.v(), kk, out);
  check_launch("k_csr_right_sparse");
}

}  // namespace skema
