// FP64 products with rows of the Gaussian RBF matrix: K_w (rows x n) is formed
// a range of points at a time into scratch memory and multiplied from there by
// the FP64 GEMM.
//   left : X       <- nu X + eta * Upsilon[:, idx] K_w     (k x n)
//   right: [y | G]  =  K_w [Omega; Psi]^T                   (w x (k+s))
// K costs 2 d + about 40 (exp) operations an element to form and 16 bytes of
// traffic a use, the products 2 (2k + s): at k = 201, s = 403 the bytes of writing
// K once and reading it twice take 1/15 of the products' time at the copy rate,
// forming K and all 12%.  Generating K inside each
// product's own tile loop instead (no K in memory) kept the product at 21 to 43
// TF, because the Gram, the exponentials and their barriers stood between its
// MFMAs, and formed K twice; here both products run at the GEMM's 58 to 64 TF.
// Window of 2048 rows, 20011 points in d = 64, k = 201, s = 403: 2.29 -> 1.36 ms
// (K 0.16, left 0.35, right 0.84).
#include "rbf_tiles.hpp"

#include <algorithm>
#include <memory>

#include "rbf.hpp"
#include "util.hpp"

namespace skema {
namespace {

constexpr int kThreads = 512;
constexpr int kTile = 128;    // rows and points of a tile
constexpr int kBF = 16;       // features per slice
constexpr int kPitch = 144;   // 16 mod 32 doubles: fragment reads touch every bank

__device__ __forceinline__ int xcd_remap(int bid, int nb) {
  const int q = nb >> 3, r = nb & 7;
  const int xcd = bid & 7, local = bid >> 3;
  return xcd * q + (xcd < r ? xcd : r) + local;
}

struct TileArgs {
  const double* X;
  int64_t n, ldp;
  int d;
  const double* nrm;
  double gamma;
  int64_t row0, rows, col0, cols;
  double* C;
  int64_t ldc;
  int64_t twice;
  double* part;
  int tiles_m;
};

// A 128 x 128 tile of K: the Gram x_i.x_j over the features on the matrix cores
// (2 x 4 waves of 4 x 2 MFMA tiles, features through double-buffered LDS in
// slices of 16), then D = |x_i|^2 + |x_j|^2 - 2 x_i.x_j, clamped at 0, and
// exp(-gamma D), with K(i, i) = 1 (src/Skema_Kernel.cpp:49-74).  Formed with
// points as the A operand, so 16 lanes hold 16 consecutive rows.  Two blocks per
// CU: one's exponentials run beside the other's MFMAs.  H: multiplies what C
// holds by 2 K and sums H o D.
template <bool H>
__global__ __launch_bounds__(kThreads, 4) void k_rbf_tiles(TileArgs g) {
  __shared__ double As[2][kBF][kPitch], Bs[2][kBF][kPitch];
  __shared__ double red[kThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  const int wm = (wave & 1) * 64, wn = (wave >> 1) * 32;
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t m0 = (int64_t)(t % g.tiles_m) * kTile, n0 = (int64_t)(t / g.tiles_m) * kTile;

  // this thread stages row (and point) tid % 128, features tid / 128 + 4 e
  const int sr = tid & 127, sf = tid >> 7;
  const int64_t ri = m0 + sr < g.rows ? m0 + sr : g.rows - 1, rj = n0 + sr < g.cols ? n0 + sr : g.cols - 1;
  const double* pa = g.X + g.row0 + ri;
  const double* pb = g.X + g.col0 + rj;
  double ra[4], rb[4];
  auto gload = [&](int f0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int f = f0 + sf + 4 * e;
      const int64_t at = (int64_t)(f < g.d ? f : g.d - 1) * g.ldp;
      const double a = pa[at], b = pb[at];
      ra[e] = f < g.d ? a : 0.0;
      rb[e] = f < g.d ? b : 0.0;
    }
  };
  auto sstore = [&](int b) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      As[b][sf + 4 * e][sr] = ra[e];
      Bs[b][sf + 4 * e][sr] = rb[e];
    }
  };
  d4 acc[4][2];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) acc[x][y] = d4{0.0, 0.0, 0.0, 0.0};
  gload(0);
  sstore(0);
  __syncthreads();
  const int slices = (g.d + kBF - 1) / kBF;
  for (int s = 0; s < slices; ++s) {
    if (s + 1 < slices) gload((s + 1) * kBF);
    const int b = s & 1;
    const int steps = g.d - s * kBF >= kBF ? 4 : (g.d - s * kBF + 3) / 4;
    for (int kk = 0; kk < steps; ++kk) {
      double a[4], p[2];
#pragma unroll
      for (int x = 0; x < 4; ++x) a[x] = As[b][4 * kk + lq][wm + 16 * x + l16];
#pragma unroll
      for (int y = 0; y < 2; ++y) p[y] = Bs[b][4 * kk + lq][wn + 16 * y + l16];
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(p[y], a[x], acc[x][y], 0, 0, 0);
    }
    if (s + 1 < slices) sstore(b ^ 1);
    __syncthreads();
  }

  const bool whole = m0 + kTile <= g.rows && n0 + kTile <= g.cols;
  double sum = 0.0;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int64_t i = m0 + wm + 16 * x + l16;
    const double ni = g.nrm[g.row0 + (i < g.rows ? i : g.rows - 1)];
    double* cp = g.C + i + (n0 + wn + lq) * g.ldc;
    double old[2][4];  // a strip's 8 values of C asked for together (and no further strip's: registers)
    if (H) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int64_t j = n0 + wn + 16 * y + lq + 4 * v;
          old[y][v] = g.C[(i < g.rows ? i : g.rows - 1) + (j < g.cols ? j : g.cols - 1) * g.ldc];
        }
    }
    double kv[2][4];
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t j = n0 + wn + 16 * y + lq + 4 * v;
        const double nj = g.nrm[g.col0 + (j < g.cols ? j : g.cols - 1)];
        double D = ni + nj - 2.0 * acc[x][y][v];
        const bool diag = g.row0 + i == g.col0 + j;
        D = D > 0.0 && !diag ? D : 0.0;
        const double e = exp(-g.gamma * D);
        kv[y][v] = diag ? 1.0 : e;
        if (H) {
          kv[y][v] *= 2.0 * old[y][v];
          const double h = kv[y][v] * D;
          sum += whole || (i < g.rows && j < g.cols) ? (j >= g.twice ? 2.0 : 1.0) * h : 0.0;
        }
      }
    if (whole) {
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int v = 0; v < 4; ++v) cp[(16 * y + 4 * v) * g.ldc] = kv[y][v];
    } else {
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (i < g.rows && n0 + wn + 16 * y + lq + 4 * v < g.cols) cp[(16 * y + 4 * v) * g.ldc] = kv[y][v];
    }
  }
  if (H) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    if (tid == 0) {
      double v = 0.0;
#pragma unroll
      for (int w = 0; w < kThreads / 64; ++w) v += red[w];
      g.part[blockIdx.x] = v;
    }
  }
}

}  // namespace

int64_t rbf_tile_blocks(int64_t rows, int64_t cols) { return cdiv(rows, kTile) * cdiv(cols, kTile); }

void rbf_tiles_f64(hipStream_t st, const RbfRows& w, int64_t col0, int64_t cols, double* C, int64_t ldc, int64_t twice,
                   double* part) {
  SKEMA_REQUIRE(w.d >= 1 && w.d <= kRbfMaxFeat, kErrUnsupported, "RBF tiles: d above 128");
  SKEMA_REQUIRE(w.rows > 0 && cols > 0 && ldc >= w.rows && w.ldp >= w.n && w.row0 >= 0 && w.row0 + w.rows <= w.n &&
                    col0 >= 0 && col0 + cols <= w.n,
                kErrShape, "RBF tiles: bad range");
  const int64_t blocks = rbf_tile_blocks(w.rows, cols);
  SKEMA_REQUIRE(blocks < (int64_t)1 << 31, kErrShape, "RBF tiles: too many");
  TileArgs a{w.X, w.n, w.ldp, (int)w.d, w.nrm, w.gamma, w.row0, w.rows, col0, cols, C, ldc, twice, part,
             (int)cdiv(w.rows, kTile)};
  if (part) hipLaunchKernelGGL((k_rbf_tiles<true>), dim3((unsigned)blocks), dim3(kThreads), 0, st, a);
  else hipLaunchKernelGGL((k_rbf_tiles<false>), dim3((unsigned)blocks), dim3(kThreads), 0, st, a);
  check_launch("k_rbf_tiles");
}

int64_t reserve_columns(DevBuf& buf, int64_t ld, int64_t n, int64_t unit, size_t most) {
  for (;;) {
    int64_t nc = std::max<int64_t>(unit, (int64_t)(most / sizeof(double)) / ld / unit * unit);
    if (nc >= n) nc = cdiv(n, unit) * unit;
    else nc = cdiv(cdiv(n, cdiv(n, nc)), unit) * unit;  // nearly equal ranges
    try {
      buf.reserve((size_t)ld * nc * sizeof(double));
      return nc;
    } catch (const Error& e) {
      if (e.code != kErrOom || nc <= unit) throw;
      (void)hipGetLastError();
      most /= 2;
    }
  }
}

void rbf_products_f64(Ctx* c, const RbfRows& w, const double* U, int64_t ldu, int64_t k, const GemmOut& left,
                      const double* OP, int64_t ldop, int64_t N, const GemmOut& right, bool timed) {
  hipStream_t st = c->stream;
  auto scope = [&](const char* name) { return timed ? std::make_unique<Timed>(c, name) : nullptr; };
  // 16 doubles past a multiple of 16: columns start on 128-byte lines, not all
  // in the same L2 channel.  1 GiB holds 2048 rows of 65536 points.
  const int64_t ld = cdiv(w.rows, 16) * 16 + 16;
  const int64_t nc = reserve_columns(c->kwin, ld, w.n, kTile, (size_t)1 << 30);
  double* K = c->kwin.as<double>();
  for (int64_t j0 = 0; j0 < w.n; j0 += nc) {
    const int64_t cols = std::min(nc, w.n - j0);
    {
      auto t = scope("window");
      rbf_tiles_f64(st, w, j0, cols, K, ld, 0, nullptr);
    }
    if (U) {
      auto t = scope("rbf_left");
      GemmOut o = left;
      o.C1 = left.C1 + j0 * left.ldc1;
      o.C2 = o.C1;
      o.nsplit = cols;
      gemm_f64(st, 'N', 'N', k, cols, w.rows, U, ldu, K, ld, o, &c->gws);
    }
    if (OP) {
      auto t = scope("rbf_right");
      GemmOut o = right;
      if (j0) o.beta1 = o.beta2 = 1.0;  // later ranges add to the first
      gemm_f64(st, 'N', 'T', w.rows, N, cols, K, ld, OP + j0 * ldop, ldop, o, &c->gws);
    }
  }
}

bool rbf_tiles_supported(const Sketch& sk) {
  return !sk.sparse_maps && sk.p.precision == SKEMA_PREC_FP64 && sk.p.nfeat >= 1 && sk.p.nfeat <= kRbfMaxFeat;
}

void update_rbf_window_tiles(Sketch& sk, const double* points, int64_t ldp, int64_t row0, int64_t rows,
                             bool have_norms) {
  Ctx* c = sk.ctx;
  hipStream_t st = c->stream;
  const int64_t k = sk.k, s = sk.s, m = sk.p.m, n = sk.p.n;
  const double eta = sk.p.eta, nu = sk.p.nu;
  sk.G.reserve((size_t)rows * s * sizeof(double));
  double* G = sk.G.as<double>();
  if (!have_norms) {
    Timed t(c, "window");
    sk.win.reserve((size_t)n * sizeof(double));
    row_norms2(st, points, n, sk.p.nfeat, ldp, sk.win.as<double>());
  }
  RbfRows w;
  w.X = points; w.n = n; w.ldp = ldp; w.d = sk.p.nfeat; w.nrm = sk.win.as<double>(); w.gamma = sk.p.gamma;
  w.row0 = row0; w.rows = rows;
  GemmOut x, y;
  x.C1 = sk.X.as<double>(); x.ldc1 = k; x.alpha1 = eta; x.beta1 = nu;
  x.ldc2 = k;
  y.C1 = sk.Y.as<double>() + row0; y.ldc1 = m; y.alpha1 = eta; y.beta1 = nu; y.nsplit = k;
  y.C2 = G; y.ldc2 = rows; y.alpha2 = 1.0; y.beta2 = 0.0;
  rbf_products_f64(c, w, sk.upsL + row0 * sk.ldups, sk.ldups, k, x, sk.omps.as<double>(), k + s, k + s, y, true);
  {
    Timed t(c, "sketch_core");
    gemm_f64(st, 'N', 'N', s, s, rows, eta, sk.phiL + row0 * sk.ldphi, sk.ldphi, G, rows, nu, sk.Z.as<double>(), s,
             &c->gws);
  }
}

}  // namespace skema
