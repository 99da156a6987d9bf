// FP64 GEMM on v_mfma_f64_16x16x4_f64 for gfx950.
//
// Operands are column-major with arbitrary leading dimension; transposition is
// a template parameter, so every global load runs along the contiguous index.
//
// MFMA 16x16x4 f64 lane layout (64 lanes, l = lane):
//   A operand  A[i][k]  with i = l % 16, k = l / 16
//   B operand  B[k][j]  with j = l % 16, k = l / 16
//   D result   D[i][j]  with j = l % 16, i = l / 16 + 4 * v, v = 0..3
//              (rows interleave by 4 across the four accumulator registers)
// The product is formed transposed (op(B)^T as the A operand, op(A)^T as the B
// operand), so a lane's four results lie in four columns of C and 16 lanes
// hold 16 consecutive rows: C is read and written in 128-byte runs.
//
// Two kernels.  k_gemm_wide: one 8-wave block per CU on a 256 x 128 tile, for
// products with enough tiles (or K to split) to fill the chip.
// k_gemm_ksplit: 32 x 32 tiles whose 2, 8 or 16 waves split K, for small products.
#include "gemm.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace skema {
namespace {

// two doubles on an 8-byte boundary
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

constexpr int kBK = 16;
constexpr int kWideThreads = 512;
constexpr int kCUs = 256;

struct KArgs {
  int64_t M, N, K;
  const double* A;
  int64_t lda;
  const double* B;
  int64_t ldb;
  GemmOut out;
  int64_t k_per_split;
  double* partial;  // split-K slices [z][M x N], nullptr -> direct epilogue
  int tiles_t, tiles_s;
  // k_gemm_ksplit<..., true>: `chain` products one after the other into the same output,
  // A and B stepA and stepB elements further each time (blockIdx.y = 0), or
  // as many products as gridDim.y, each into its own output
  int chain = 1;
  int64_t stepA = 0, stepB = 0, stepC1 = 0, stepC2 = 0;
};

// Workgroup ids are dealt round-robin to the 8 XCDs; give each XCD a
// contiguous range of tiles so neighbouring tiles share that XCD's L2.
__device__ __forceinline__ int xcd_remap(int bid, int nb) {
  const int q = nb >> 3, r = nb & 7;
  const int xcd = bid & 7, local = bid >> 3;
  return xcd * q + (xcd < r ? xcd : r) + local;
}

__device__ __forceinline__ void store_out(const GemmOut& o, int64_t i, int64_t j, double v) {
  if (j < o.nsplit) {
    double* c = o.C1 + i + j * o.ldc1;
    *c = (o.beta1 != 0.0) ? o.alpha1 * v + o.beta1 * *c : o.alpha1 * v;
  } else {
    double* c = o.C2 + i + (j - o.nsplit) * o.ldc2;
    *c = (o.beta2 != 0.0) ? o.alpha2 * v + o.beta2 * *c : o.alpha2 * v;
  }
}

// Barrier after this wave's LDS accesses have completed.  Unlike
// __syncthreads it leaves global loads in flight.
__device__ __forceinline__ void lds_sync() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// LDS image of a ROWS x 16 operand slice.  Operands whose rows are contiguous
// in memory are kept [k][row] with a pitch of 16 mod 32 doubles, K-contiguous
// ones [row][k] with a pitch of 18: either way the 64 lanes of a fragment
// read (16 rows x 4 k) and of a staging write touch every bank evenly.
template <bool KC, int ROWS>
struct Slice {
  static constexpr int P = KC ? kBK + 2 : (ROWS % 32 == 16 ? ROWS : ROWS + 16);
  static constexpr int SIZE = KC ? ROWS * P : kBK * P;
  static constexpr int E = (ROWS * kBK + kWideThreads - 1) / kWideThreads;  // staged doubles per thread
  static constexpr bool EVEN = ROWS * kBK % kWideThreads == 0;
  static __device__ __forceinline__ int at(int k, int r) { return KC ? r * P + k : k * P + r; }
  // staged element idx is (k_of, r_of); threads past the end load the last one again
  static __device__ __forceinline__ int clip(int idx) { return EVEN || idx < ROWS * kBK ? idx : ROWS * kBK - 1; }
  static __device__ __forceinline__ int k_of(int idx) { return KC ? idx % kBK : idx / ROWS; }
  static __device__ __forceinline__ int r_of(int idx) { return KC ? idx / kBK : idx % ROWS; }
};

// One block tile: WM x (8 / WM) waves, each TM x TN MFMA tiles.  What bounds
// the path is the FP64 matrix rate (64 cycles per MFMA and SIMD): a slice of 16
// is 512 TM TN cycles per SIMD, against which the LDS reads (128 (TM + TN)
// cycles a slice) and the L2 requests (12 B a cycle and CU at 256 x 128; tiles
// of 64 x 64 asked for 32) stay hidden.  Slices are double-buffered in LDS:
// while slice t is multiplied, slice t+1 goes from registers to LDS and the
// loads of t+2 are issued, with one barrier per slice and two waves per SIMD.
// Rows past the operand read its last row (their results are not stored);
// only a last slice of fewer than 16 of K tests its elements.
// Measured: 4096 x 1204 x 16384 (NT) 3.78 -> 2.64 ms (61 TF of the 78.6 TF
// peak), 401 x 16384 x 4096 (NN) 1.35 -> 0.90 ms, 8192^3 69 TF; before, 64 x 64
// tiles of 4 waves with two barriers per slice.
// FAR: 64-bit offsets, for leading dimensions whose slices span 4 GiB or more
// (near_enough below).
template <int WM, int TM, int TN, bool TA, bool TB, bool FAR>
__device__ __forceinline__ void wide_tile(const KArgs& g, double* lds, int64_t m0, int64_t n0, int64_t m1, int64_t n1,
                                          int64_t kbeg, int64_t kend, int split) {
  constexpr int RA = WM * TM * 16, RB = (8 / WM) * TN * 16;
  using SA = Slice<TA, RA>;
  using SB = Slice<!TB, RB>;
  constexpr int BUF = SA::SIZE + SB::SIZE;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  const int wm = WM == 8 ? wave : 0, wn = WM == 8 ? 0 : wave;

  using Off = std::conditional_t<FAR, uint64_t, uint32_t>;
  Off oa[SA::E], ob[SB::E];  // byte offsets from the slice's first element
#pragma unroll
  for (int e = 0; e < SA::E; ++e) {
    const int idx = SA::clip(tid + e * kWideThreads);
    const int64_t last = g.M - 1 - m0;
    const int64_t r = SA::r_of(idx) < last ? SA::r_of(idx) : last;
    oa[e] = (Off)((TA ? SA::k_of(idx) + r * g.lda : r + SA::k_of(idx) * g.lda) * 8);
  }
#pragma unroll
  for (int e = 0; e < SB::E; ++e) {
    const int idx = SB::clip(tid + e * kWideThreads);
    const int64_t last = g.N - 1 - n0;
    const int64_t r = SB::r_of(idx) < last ? SB::r_of(idx) : last;
    ob[e] = (Off)((TB ? r + SB::k_of(idx) * g.ldb : SB::k_of(idx) + r * g.ldb) * 8);
  }
  const char* pa = reinterpret_cast<const char*>(g.A + (TA ? m0 * g.lda + kbeg : m0 + kbeg * g.lda));
  const char* pb = reinterpret_cast<const char*>(g.B + (TB ? n0 + kbeg * g.ldb : n0 * g.ldb + kbeg));
  const int64_t stepa = (TA ? kBK : kBK * g.lda) * 8, stepb = (TB ? kBK * g.ldb : kBK) * 8;

  double ra[SA::E], rb[SB::E];
  constexpr int NS = SA::E + SB::E;  // staged doubles per thread
  auto gload1 = [&](const char* qa, const char* qb, int e) {
    if (e < SA::E) ra[e] = *reinterpret_cast<const double*>(qa + oa[e]);
    else rb[e - SA::E] = *reinterpret_cast<const double*>(qb + ob[e - SA::E]);
  };
  auto gload = [&](int64_t t) {  // slice t, all 16 of K present
#pragma unroll
    for (int e = 0; e < NS; ++e) gload1(pa + t * stepa, pb + t * stepb, e);
  };
  auto gload_tail = [&](int64_t t, int left) {  // the last slice, left < 16 of K (past it: its first, then 0)
    const char* qa = pa + t * stepa;
    const char* qb = pb + t * stepb;
#pragma unroll
    for (int e = 0; e < SA::E; ++e) {
      const int k = SA::k_of(SA::clip(tid + e * kWideThreads));
      const Off back = k < left ? 0 : (Off)(k * (TA ? 1 : g.lda) * 8);
      const double v = *reinterpret_cast<const double*>(qa + (oa[e] - back));
      ra[e] = k < left ? v : 0.0;
    }
#pragma unroll
    for (int e = 0; e < SB::E; ++e) {
      const int k = SB::k_of(SB::clip(tid + e * kWideThreads));
      const Off back = k < left ? 0 : (Off)(k * (TB ? g.ldb : 1) * 8);
      const double v = *reinterpret_cast<const double*>(qb + (ob[e] - back));
      rb[e] = k < left ? v : 0.0;
    }
  };
  auto sstore1 = [&](int b, int e) {
    double* As = lds + b * BUF;
    if (e < SA::E) {
      const int idx = tid + e * kWideThreads;
      if (SA::EVEN || idx < RA * kBK) As[SA::at(SA::k_of(idx), SA::r_of(idx))] = ra[e];
    } else {
      const int idx = tid + (e - SA::E) * kWideThreads;
      if (SB::EVEN || idx < RB * kBK) As[SA::SIZE + SB::at(SB::k_of(idx), SB::r_of(idx))] = rb[e - SA::E];
    }
  };
  auto sstore = [&](int b) {
#pragma unroll
    for (int e = 0; e < NS; ++e) sstore1(b, e);
  };

  d4 acc[TM][TN];
#pragma unroll
  for (int x = 0; x < TM; ++x)
#pragma unroll
    for (int y = 0; y < TN; ++y) acc[x][y] = d4{0.0, 0.0, 0.0, 0.0};

  // Fragment f of K step kk of the slice in buffer b.
  auto frag1 = [&](int b, int kk, int f, double (&fa)[TM], double (&fb)[TN]) {
    const double* As = lds + b * BUF;
    if (f < TM) fa[f] = As[SA::at(4 * kk + lq, (wm * TM + f) * 16 + l16)];
    else fb[f - TM] = As[SA::SIZE + SB::at(4 * kk + lq, (wn * TN + f - TM) * 16 + l16)];
  };
  auto frags = [&](int b, int kk, double (&fa)[TM], double (&fb)[TN]) {
#pragma unroll
    for (int f = 0; f < TM + TN; ++f) frag1(b, kk, f, fa, fb);
  };
  // The MFMAs of one K step with `others` further instructions dealt out
  // evenly among them (other(i), i < others); the scheduling fences keep them
  // there, so that a wave's loads and LDS accesses issue while the matrix core
  // is busy.  In one run they left it idle 17% of the cycles, because the two
  // waves of a SIMD come to them together.
  auto mma = [&](const double (&fa)[TM], const double (&fb)[TN], auto others, auto&& other) {
    constexpr int NM = TM * TN, NO = decltype(others)::value;
#pragma unroll
    for (int q = 0; q < NM; ++q) {
      const int x = q / TN, y = q % TN;
      acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[y], fa[x], acc[x][y], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = q * NO / NM; i < (q + 1) * NO / NM; ++i) other(i);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Whole slices without a branch: past the last one the loads repeat it and
  // what is staged and read from it is not used.  Each K step's fragments are
  // read while the step before is multiplied; the barrier stands before the
  // slice's last step, whose fragments are in registers by then, so the next
  // slice's first reads run under MFMAs too and no wave reads the buffer that
  // the next slice's staging overwrites.
  const int64_t full = (kend - kbeg) / kBK;
  const int left = (int)((kend - kbeg) % kBK);
  constexpr int NF = TM + TN;
  double a0[TM], b0[TN], a1[TM], b1[TN];
  if (full > 0) {
    gload(0);
    sstore(0);
    gload(full > 1 ? 1 : 0);
    lds_sync();
    frags(0, 0, a0, b0);
    for (int64_t t = 0; t < full; ++t) {
      const int b = (int)(t & 1);
      const int64_t tn = t + 2 < full ? t + 2 : full - 1;
      const char* qa = pa + tn * stepa;
      const char* qb = pb + tn * stepb;
      mma(a0, b0, std::integral_constant<int, NF>{}, [&](int i) { frag1(b, 1, i, a1, b1); });
      mma(a1, b1, std::integral_constant<int, NF + 2 * NS>{}, [&](int i) {
        if (i < NF) {
          frag1(b, 2, i, a0, b0);
        } else if ((i - NF) % 2 == 0) {  // slice t + 1 out of a register, then slice t + 2 into it
          sstore1(b ^ 1, (i - NF) / 2);
        } else {
          gload1(qa, qb, (i - NF) / 2);
        }
      });
      mma(a0, b0, std::integral_constant<int, NF>{}, [&](int i) { frag1(b, 3, i, a1, b1); });
      lds_sync();
      mma(a1, b1, std::integral_constant<int, NF>{}, [&](int i) { frag1(b ^ 1, 0, i, a0, b0); });
    }
  }
  if (left > 0) {
    lds_sync();  // the last reads of buffer full & 1, above, are done
    const int b = (int)(full & 1);
    gload_tail(full, left);
    sstore(b);
    lds_sync();
    for (int kk = 0; 4 * kk < left; ++kk) {
      frags(b, kk, a0, b0);
      mma(a0, b0, std::integral_constant<int, 0>{}, [](int) {});
    }
  }

  // Epilogue, one 16-row strip at a time: all of its old values are asked for
  // before the first is used (rows and columns past the end read the last).
  const bool keep = !g.partial && (g.out.beta1 != 0.0 || g.out.beta2 != 0.0);
#pragma unroll
  for (int x = 0; x < TM; ++x) {
    const int64_t i = m0 + (wm * TM + x) * 16 + l16;
    const int64_t j0 = n0 + wn * TN * 16 + lq;
    double old[TN][4];
    if (keep) {
      const int64_t ic = i < m1 ? i : m1 - 1;
#pragma unroll
      for (int y = 0; y < TN; ++y)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int64_t j = j0 + 16 * y + 4 * v, jc = j < n1 ? j : n1 - 1;
          const double* c = jc < g.out.nsplit ? g.out.C1 + jc * g.out.ldc1 : g.out.C2 + (jc - g.out.nsplit) * g.out.ldc2;
          old[y][v] = c[ic];
        }
    }
#pragma unroll
    for (int y = 0; y < TN; ++y)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t j = j0 + 16 * y + 4 * v;
        if (i < m1 && j < n1) {
          double r = acc[x][y][v];
          if (g.partial) {
            g.partial[(int64_t)split * g.M * g.N + i + j * g.M] = r;
          } else {
            const bool first = j < g.out.nsplit;
            double* c = first ? g.out.C1 + i + j * g.out.ldc1 : g.out.C2 + i + (j - g.out.nsplit) * g.out.ldc2;
            const double alpha = first ? g.out.alpha1 : g.out.alpha2, beta = first ? g.out.beta1 : g.out.beta2;
            r *= alpha;
            if (beta != 0.0) r += beta * old[y][v];
            *c = r;
          }
        }
      }
  }
}

// The eight waves lie along T (M when WM == 8, N when WM == 1), 16 TT rows of
// it each; all of them share the block's part of S, which is cut into tiles_s
// nearly equal parts of at most TS MFMA tiles (401 rows are 7 + 7 + 6 + 6
// tiles, not 8 + 8 + 8 + 2); a part below TS is multiplied as TS - 1 tiles.
template <int WM, int TT, int TS, bool TA, bool TB, bool FAR>
__global__ __launch_bounds__(kWideThreads) void k_gemm_wide(KArgs g) {
  constexpr int RT = 8 * TT * 16, RS = TS * 16;
  constexpr int SZ_T = WM == 8 ? Slice<TA, RT>::SIZE : Slice<!TB, RT>::SIZE;
  constexpr int SZ_S = WM == 8 ? Slice<!TB, RS>::SIZE : Slice<TA, RS>::SIZE;
  __shared__ double lds[2 * (SZ_T + SZ_S)];
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  const int ti = t / g.tiles_s, si = t % g.tiles_s;
  const int64_t ns = ((WM == 8 ? g.N : g.M) + 15) / 16;
  const int64_t s0 = si * ns / g.tiles_s, s1 = (si + 1) * ns / g.tiles_s;
  const int64_t m0 = WM == 8 ? (int64_t)ti * RT : s0 * 16, n0 = WM == 8 ? s0 * 16 : (int64_t)ti * RT;
  const int64_t kbeg = (int64_t)blockIdx.z * g.k_per_split;
  const int64_t kend = (g.K < kbeg + g.k_per_split) ? g.K : kbeg + g.k_per_split;
  const int64_t e1 = s1 * 16;
  const int64_t m1 = WM == 8 || e1 > g.M ? g.M : e1, n1 = WM == 8 && e1 < g.N ? e1 : g.N;
  if constexpr (TS == 1) {
    wide_tile<WM, WM == 8 ? TT : 1, WM == 8 ? 1 : TT, TA, TB, FAR>(g, lds, m0, n0, m1, n1, kbeg, kend, blockIdx.z);
  } else {
    if (s1 - s0 == TS)
      wide_tile<WM, WM == 8 ? TT : TS, WM == 8 ? TS : TT, TA, TB, FAR>(g, lds, m0, n0, m1, n1, kbeg, kend,
                                                                      blockIdx.z);
    else
      wide_tile<WM, WM == 8 ? TT : TS - 1, WM == 8 ? TS - 1 : TT, TA, TB, FAR>(g, lds, m0, n0, m1, n1, kbeg, kend,
                                                                              blockIdx.z);
  }
}

// Small products: a 32 x 32 tile per block, K dealt to its KW waves in
// chunks of 16, operands straight from global memory into MFMA fragments (the
// next two chunks' loads in flight while this one is multiplied), the KW
// partial tiles summed through LDS in wave order.  These products are bound by
// the latency of their K loop: 64 x 98 x 300 took 26 us with 64 x 64 tiles and a
// barrier pair per 16 of K, and takes 5 us here; 803 x 803 x 4096 124 us.
template <int KW, bool TA, bool TB, bool SERIES = false>
__global__ __launch_bounds__(64 * KW) void k_gemm_ksplit(KArgs g) {
  __shared__ double part[KW][32][33];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  const int64_t m0 = (int64_t)(blockIdx.x % g.tiles_t) * 32, n0 = (int64_t)(blockIdx.x / g.tiles_t) * 32;
  const int64_t kbeg = (int64_t)blockIdx.z * g.k_per_split;
  const int64_t kend = (g.K < kbeg + g.k_per_split) ? g.K : kbeg + g.k_per_split;
  const int64_t sa = TA ? 1 : g.lda, sb = TB ? g.ldb : 1;
  const double* pa[2];
  const double* pb[2];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    int64_t i = m0 + 16 * x + l16, j = n0 + 16 * x + l16;
    i = i < g.M ? i : g.M - 1;  // rows past the end: results not stored
    j = j < g.N ? j : g.N - 1;
    pa[x] = g.A + (SERIES ? blockIdx.y * g.stepA : 0) + (TA ? i * g.lda : i) + (kbeg + 2 * lq) * sa;
    pb[x] = g.B + (SERIES ? blockIdx.y * g.stepB : 0) + (TB ? j : j * g.ldb) + (kbeg + 2 * lq) * sb;
  }
  GemmOut out = g.out;
  if (SERIES) {
    out.C1 += blockIdx.y * g.stepC1;
    out.C2 += blockIdx.y * g.stepC2;
  }
  d4 acc[2][2];
  struct Frags {
    double a[2][4], b[2][4];
  };
  // K step kk of a chunk multiplies k = 8 (kk / 2) + 2 lq + kk % 2, so a
  // K-contiguous operand comes in pairs: 64 bytes of a row per load, not 32.
  auto load = [&](Frags& f, int64_t c) {  // chunk c, all 16 of K present
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const double* qa = pa[x] + (16 * c + 8 * h) * sa;
        const double* qb = pb[x] + (16 * c + 8 * h) * sb;
        if (TA) {
          const d2u v = *reinterpret_cast<const d2u*>(qa);
          f.a[x][2 * h] = v.x;
          f.a[x][2 * h + 1] = v.y;
        } else {
          f.a[x][2 * h] = qa[0];
          f.a[x][2 * h + 1] = qa[sa];
        }
        if (!TB) {
          const d2u v = *reinterpret_cast<const d2u*>(qb);
          f.b[x][2 * h] = v.x;
          f.b[x][2 * h + 1] = v.y;
        } else {
          f.b[x][2 * h] = qb[0];
          f.b[x][2 * h + 1] = qb[sb];
        }
      }
  };
  auto mma = [&](const Frags& f) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.b[y][kk], f.a[x][kk], acc[x][y], 0, 0, 0);
  };
  // this wave's whole chunks: wave, wave + KW, ...
  const int64_t full = (kend - kbeg) / 16;
  const int left = (int)((kend - kbeg) % 16);
  Frags f0, f1;
  for (int link = 0; link < (SERIES ? g.chain : 1); ++link) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) acc[x][y] = d4{0.0, 0.0, 0.0, 0.0};
    if (wave < full) {
      int64_t n = (full - 1 - wave) / KW + 1;
      const int64_t last = wave + (n - 1) * KW;
      auto at = [&](int64_t c) { return c < last ? c : last; };
      int64_t c = wave;
      load(f0, c);
      load(f1, at(c + KW));
      for (; n > 1; n -= 2) {
        mma(f0);
        load(f0, at(c + 2 * KW));
        mma(f1);
        load(f1, at(c + 3 * KW));
        c += 2 * KW;
      }
      if (n) mma(f0);
    }
    if (left > 0 && wave == (int)(full % KW)) {
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const int kc = 8 * (kk / 2) + kk % 2;
        const bool ok = kc + 2 * lq < left;
        const int64_t k = 16 * full + (ok ? kc : -2 * lq);  // else this chunk's first
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const double va = pa[x][k * sa], vb = pb[x][k * sb];
          f0.a[x][kk] = ok ? va : 0.0;
          f0.b[x][kk] = ok ? vb : 0.0;
        }
      }
      mma(f0);
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int v = 0; v < 4; ++v) part[wave][16 * y + lq + 4 * v][16 * x + l16] = acc[x][y][v];
    __syncthreads();
#pragma unroll
    for (int e = tid; e < 1024; e += 64 * KW) {
      const int ii = e & 31, jj = e >> 5;
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < KW; ++w) s += part[w][jj][ii];
      const int64_t i = m0 + ii, j = n0 + jj;
      if (i < g.M && j < g.N) {
        if (g.partial) g.partial[(int64_t)blockIdx.z * g.M * g.N + i + j * g.M] = s;
        else store_out(out, i, j, s);
      }
    }
    if (SERIES && link + 1 < g.chain) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        pa[x] += g.stepA;
        pb[x] += g.stepB;
      }
      __syncthreads();  // the partial tiles have been read
    }
  }
}

// Deterministic split-K reductions.  Large outputs: one element per thread, the
// slices added in order.  Bound by reading the partials: 59 MB (6 slices of
// 2048 x 604) took 52 us in the other form.
__global__ __launch_bounds__(256) void k_splitk_sum(const double* part, int splits, int64_t M, int64_t total, GemmOut o) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= total) return;
  double s = 0.0;
#pragma unroll 4
  for (int z = 0; z < splits; ++z) s += part[(int64_t)z * total + e];
  const int64_t j = total < (int64_t)1 << 32 ? (int64_t)((uint32_t)e / (uint32_t)M) : e / M;
  store_out(o, e - j * M, j, s);
}
// Small outputs: 32 consecutive elements x 8 groups of slices per block (group q
// sums slices q, q + 8, ... in order, then the groups are added in order), so
// many slices of a small product are read by many threads.
__global__ __launch_bounds__(256) void k_splitk_reduce(const double* part, int splits, int64_t M, int64_t total,
                                                       GemmOut o) {
  __shared__ double red[8][33];
  const int tid = threadIdx.x, c = tid & 31, q = tid >> 5;
  for (int64_t e0 = (int64_t)blockIdx.x * 32; e0 < total; e0 += (int64_t)gridDim.x * 32) {
    const int64_t e = e0 + c;
    double s = 0.0;
    if (e < total)
      for (int z = q; z < splits; z += 8) s += part[(int64_t)z * total + e];
    red[q][c] = s;
    __syncthreads();
    if (q == 0 && e < total) {
      double v = 0.0;
#pragma unroll
      for (int w = 0; w < 8; ++w) v += red[w][c];
      store_out(o, e % M, e / M, v);
    }
    __syncthreads();
  }
}

template <int WM, int TT, int TS, bool FAR>
void launch_wide_t(hipStream_t st, bool ta, bool tb, const KArgs& a, dim3 grid) {
  const dim3 block(kWideThreads);
  if (!ta && !tb) hipLaunchKernelGGL((k_gemm_wide<WM, TT, TS, false, false, FAR>), grid, block, 0, st, a);
  else if (!ta && tb) hipLaunchKernelGGL((k_gemm_wide<WM, TT, TS, false, true, FAR>), grid, block, 0, st, a);
  else if (ta && !tb) hipLaunchKernelGGL((k_gemm_wide<WM, TT, TS, true, false, FAR>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((k_gemm_wide<WM, TT, TS, true, true, FAR>), grid, block, 0, st, a);
}
template <int WM, int TT, bool FAR>
void launch_wide_s(hipStream_t st, bool ta, bool tb, const KArgs& a, dim3 grid, int ts) {
  if (ts == 8) launch_wide_t<WM, TT, 8, FAR>(st, ta, tb, a, grid);
  else if (ts >= 6) launch_wide_t<WM, TT, 7, FAR>(st, ta, tb, a, grid);
  else if (ts >= 4) launch_wide_t<WM, TT, 5, FAR>(st, ta, tb, a, grid);
  else if (ts >= 2) launch_wide_t<WM, TT, 3, FAR>(st, ta, tb, a, grid);
  else launch_wide_t<WM, TT, 1, FAR>(st, ta, tb, a, grid);
}

template <int KW>
void launch_ksplit(hipStream_t st, bool ta, bool tb, const KArgs& a, dim3 grid) {
  const dim3 block(64 * KW);
  if (!ta && !tb) hipLaunchKernelGGL((k_gemm_ksplit<KW, false, false>), grid, block, 0, st, a);
  else if (!ta && tb) hipLaunchKernelGGL((k_gemm_ksplit<KW, false, true>), grid, block, 0, st, a);
  else if (ta && !tb) hipLaunchKernelGGL((k_gemm_ksplit<KW, true, false>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((k_gemm_ksplit<KW, true, true>), grid, block, 0, st, a);
}

template <int KW>
void launch_series(hipStream_t st, bool tb, const KArgs& a, dim3 grid) {
  if (tb) hipLaunchKernelGGL((k_gemm_ksplit<KW, false, true, true>), grid, dim3(64 * KW), 0, st, a);
  else hipLaunchKernelGGL((k_gemm_ksplit<KW, false, false, true>), grid, dim3(64 * KW), 0, st, a);
}

// One way to run a product, with its estimated time in CU cycles.
struct Plan {
  bool wide = false, far = false;
  int wm = 8;  // wide: waves along M (8) or N (1); else the block's waves
  int tt = 2, ts = 8, splits = 1;
  int64_t tiles_t = 1, tiles_s = 1;
  double cost = 1e300;
};

// Estimated cycles of the wide kernel: rounds of 256 blocks, a slice costing
// the most of its MFMA, LDS and L2 time, plus writing and reading the K
// splits' partials at about 4 TB/s and the launch that adds them.  The partials
// stay within most_bytes.
// far: the 64-bit form, built for TT = 2 only.
// K of at most kShortK: the rounds' stores run beside the products of other
// blocks and bound most of these, at 1785 B a cycle; blocks whose waves hold 128
// rows of a column (WM = 1, TT = 1) write the longest runs.  14919 x 3410 x 6
// takes 115 us with those, 121 with WM = 8, 158 with TT = 2 and 203 with both.
constexpr int64_t kShortK = 128;
void try_wide(Plan& best, int64_t M, int64_t N, int64_t K, size_t most_bytes, bool far) {
  const int64_t room = (int64_t)(most_bytes / sizeof(double)) / (M * N);  // splits whose partials fit
  for (int wm : {8, 1}) {
    const int64_t T = wm == 8 ? M : N, ns = cdiv(wm == 8 ? N : M, 16);
    for (int tt : {2, 1}) {
      if (far && tt == 1) continue;
      const int64_t tiles_t = cdiv(T, 128 * tt), tiles_s = cdiv(ns, 8);
      if (tiles_t * tiles_s >= (int64_t)1 << 31) continue;
      const int ts = (int)cdiv(ns, tiles_s);
      const double rows = 128.0 * tt + 16.0 * ts;
      const double slice = 600.0 + std::max({512.0 * tt * ts, 128.0 * (tt + ts) + rows, rows * 128.0 / 12.0});
      if (K <= kShortK) {
        const double out = (double)M * (double)N * 8.0 / 1785.0;
        const double runs = tt == 1 ? (wm == 1 ? 1.0 : 1.05) : (wm == 1 ? 1.1 : 1.4);
        const double cost = (double)cdiv(tiles_t * tiles_s, kCUs) * (double)cdiv(K, kBK) * slice + 5000.0 +
                            std::max(40.0 * tt * ts, out * runs);
        if (cost < best.cost) best = Plan{true, far, wm, tt, ts, 1, tiles_t, tiles_s, cost};
        continue;
      }
      const int64_t most = std::max<int64_t>(1, std::min<int64_t>({128, K / 64, room}));
      for (int64_t sp = 1; sp <= most; ++sp) {
        const int64_t per = cdiv(cdiv(K, sp), kBK) * kBK;
        const int64_t real = per ? cdiv(K, per) : 1;
        if (real != sp) continue;
        const double rounds = (double)cdiv(tiles_t * tiles_s * sp, kCUs);
        double cost = rounds * ((double)(per / kBK) * slice + 5000.0 + 40.0 * tt * ts);
        if (sp > 1) cost += 8000.0 + 16.0 * (double)sp * (double)M * (double)N / 1700.0;
        if (cost < best.cost) best = Plan{true, far, wm, tt, ts, (int)sp, tiles_t, tiles_s, cost};
      }
    }
  }
}
// The same for the small kernel, with 16 waves a block while that leaves one
// block per CU and 8 otherwise.  A block's chunks (16 of K for each of its
// waves) are bound by the latency of their loads, by its MFMAs (1024 cycles per
// 4 waves) or, with more than one block per CU, by the loads' L1 traffic.
// K of at most kShortK gives a wave one chunk or none, and several blocks run on
// a CU at once: 2 waves a block there, or 8 while their blocks are few.  Measured,
// before (wide or 8 waves) and after: 694 x 454 x 32 12.7 -> 6.9 us, 439 x 1788 x 76
// 18 -> 9.9, 1457 x 5553 x 14 36 -> 28 (with the wide kernel's rule above).
// From 8192 of K on, both operands contiguous along K (TN) ask for them in
// half lines, at 2700 B a cycle once 32 tiles do so: 403 x 403 x 20000 is 278 us
// of that, and 164 on the wide kernel.
void try_ksplit(Plan& best, bool tn_form, int64_t M, int64_t N, int64_t K, size_t most_bytes) {
  const int64_t tm = cdiv(M, 32), tn = cdiv(N, 32);
  if (tm * tn >= (int64_t)1 << 31) return;
  if (K <= kShortK) {
    const double t = (double)(tm * tn) / kCUs, k16 = (double)cdiv(K, kBK);
    const double eight = std::max(7000.0, t * (2570.0 + 330.0 * k16));
    const double two = std::max(6000.0 + 1000.0 * std::ceil(k16 / 2), t * (1170.0 + 540.0 * k16));
    if (eight < best.cost) best = Plan{false, false, 8, 1, 1, 1, tm, tn, eight};
    if (two < best.cost) best = Plan{false, false, 2, 1, 1, 1, tm, tn, two};
    return;
  }
  const int64_t room = (int64_t)(most_bytes / sizeof(double)) / (M * N);
  const int64_t most = std::max<int64_t>(1, std::min<int64_t>({64, K / 512, room}));
  for (int64_t sp = 1; sp <= most; ++sp) {
    const int64_t per = cdiv(cdiv(K, sp), kBK) * kBK;
    if ((per ? cdiv(K, per) : 1) != sp) continue;
    const int64_t blocks = tm * tn * sp;
    const int kw = blocks <= kCUs && per > 16 * 8 ? 16 : 8;
    const double rounds = (double)cdiv(blocks, kCUs), chunk = kw == 16 ? 4600.0 : blocks <= kCUs ? 3000.0 : 4500.0;
    double cost = rounds * ((double)cdiv(per, 16 * kw) * chunk + 4000.0);
    if (tn_form && kw == 16 && K >= 8192 && tm * tn >= 32) cost = std::max(cost, (double)(tm * tn) * (double)K * 512.0 / 2700.0);
    if (sp > 1) cost += 8000.0 + 16.0 * (double)sp * (double)M * (double)N / 1700.0;
    if (cost < best.cost) best = Plan{false, false, kw, 1, 1, (int)sp, tm, tn, cost};
  }
}

// Whether a slice of an operand spans less than 4 GiB, 32-bit byte offsets: up to
// 256 rows ld apart where K is contiguous, 16 of K ld apart where the rows are.
// Past that the 64-bit form, at the same speed: windows of 200000 rows of a
// column-major 2200000 x 256 matrix, k = 201, s = 403 3.07 ms, as at 2000000 rows
// (5.38 on the small kernel).
bool near_enough(bool k_contiguous, int64_t ld) { return ld <= (int64_t)1 << (k_contiguous ? 21 : 25); }

// What the K splits' partials of one product may take, for the context's life:
// 8 splits of 4096 x 1204 are 316 MB; more (4 of 66000 x 604, 1.28 GB) would even
// out the last round of a product that has many.
constexpr size_t kMostPartials = (size_t)512 << 20;

Plan choose(bool ta, bool tb, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, size_t most_bytes) {
  Plan p;
  try_ksplit(p, ta && !tb, M, N, K, most_bytes);
  try_wide(p, M, N, K, most_bytes, !near_enough(ta, lda) || !near_enough(!tb, ldb));
  return p;
}

}  // namespace

bool gemm_f64_one_pass(char transB, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb) {
  if (M <= 0 || N <= 0 || K <= 0) return false;
  const Plan p = choose(false, transB == 'T' || transB == 't', M, N, K, lda, ldb, kMostPartials);
  return p.cost < 1e300 && !p.wide && p.splits == 1;
}

void gemm_f64_series(hipStream_t stream, char transB, int64_t M, int64_t N, int64_t K, const double* A,
                     int64_t lda, const double* B, int64_t ldb, const GemmOut& out, const GemmSeries& sr) {
  const bool tb = (transB == 'T' || transB == 't');
  SKEMA_REQUIRE(gemm_f64_one_pass(transB, M, N, K, lda, ldb) && sr.count > 0 && (sr.chain || sr.count <= 65535), kErrShape,
                "gemm_f64_series: not products of one pass");
  SKEMA_REQUIRE(lda >= M && ldb >= (tb ? N : K), kErrShape, "gemm_f64_series: leading dimension too small");
  Plan p;
  try_ksplit(p, false, M, N, K, kMostPartials);
  KArgs a;
  a.M = M; a.N = N; a.K = K; a.A = A; a.lda = lda; a.B = B; a.ldb = ldb; a.out = out;
  a.tiles_t = (int)p.tiles_t; a.tiles_s = (int)p.tiles_s;
  a.partial = nullptr;
  a.k_per_split = cdiv(K, kBK) * kBK;
  a.stepA = sr.stepA; a.stepB = sr.stepB; a.stepC1 = sr.stepC1; a.stepC2 = sr.stepC2;
  a.chain = sr.chain ? (int)sr.count : 1;
  const dim3 grid((unsigned)(p.tiles_t * p.tiles_s), sr.chain ? 1u : (unsigned)sr.count, 1);
  if (p.wm == 16) launch_series<16>(stream, tb, a, grid);
  else if (p.wm == 2) launch_series<2>(stream, tb, a, grid);
  else launch_series<8>(stream, tb, a, grid);
  check_launch("k_gemm_ksplit (series)");
}

void gemm_f64(hipStream_t stream, char transA, char transB, int64_t M, int64_t N, int64_t K,
              const double* A, int64_t lda, const double* B, int64_t ldb, const GemmOut& out,
              GemmWorkspace* ws) {
  SKEMA_REQUIRE(M >= 0 && N >= 0 && K >= 0, kErrShape, "gemm_f64: negative dimension");
  if (M == 0 || N == 0) return;
  const bool ta = (transA == 'T' || transA == 't');
  const bool tb = (transB == 'T' || transB == 't');
  SKEMA_REQUIRE(lda >= (ta ? (K > 0 ? K : 1) : M), kErrShape, "gemm_f64: lda too small");
  SKEMA_REQUIRE(ldb >= (tb ? N : (K > 0 ? K : 1)), kErrShape, "gemm_f64: ldb too small");
  SKEMA_REQUIRE(out.nsplit >= 0 && out.nsplit <= N, kErrArg, "gemm_f64: bad column split");
  SKEMA_REQUIRE(out.nsplit == 0 || out.ldc1 >= M, kErrShape, "gemm_f64: ldc too small");
  SKEMA_REQUIRE(out.nsplit == N || out.ldc2 >= M, kErrShape, "gemm_f64: ldc too small");
  SKEMA_REQUIRE(M * N < (int64_t)1 << 40, kErrShape, "gemm_f64: output too large");

  // Fewer splits where the device has no room for the partials.
  size_t most = ws ? kMostPartials : 0;
  Plan p;
  for (;;) {
    p = choose(ta, tb, M, N, K, lda, ldb, most);
    if (p.splits == 1) break;
    const size_t need = (size_t)p.splits * M * N * sizeof(double);
    try {
      ws->buf.reserve(need);
      break;
    } catch (const Error& e) {
      if (e.code != kErrOom) throw;
      (void)hipGetLastError();
      most = need / 2;
    }
  }
  SKEMA_REQUIRE(p.cost < 1e300, kErrShape, "gemm_f64: too many tiles");

  KArgs a;
  a.M = M; a.N = N; a.K = K; a.A = A; a.lda = lda; a.B = B; a.ldb = ldb; a.out = out;
  a.tiles_t = (int)p.tiles_t; a.tiles_s = (int)p.tiles_s;
  a.partial = nullptr;
  a.k_per_split = K > 0 ? cdiv(cdiv(K, (int64_t)p.splits), kBK) * kBK : 0;
  if (p.splits > 1) a.partial = ws->buf.as<double>();
  dim3 grid((unsigned)(p.tiles_t * p.tiles_s), 1, (unsigned)p.splits);
  if (p.wide) {
    if (p.far && p.wm == 8) launch_wide_s<8, 2, true>(stream, ta, tb, a, grid, p.ts);
    else if (p.far) launch_wide_s<1, 2, true>(stream, ta, tb, a, grid, p.ts);
    else if (p.wm == 8 && p.tt == 2) launch_wide_s<8, 2, false>(stream, ta, tb, a, grid, p.ts);
    else if (p.wm == 8) launch_wide_s<8, 1, false>(stream, ta, tb, a, grid, p.ts);
    else if (p.tt == 2) launch_wide_s<1, 2, false>(stream, ta, tb, a, grid, p.ts);
    else launch_wide_s<1, 1, false>(stream, ta, tb, a, grid, p.ts);
    check_launch("k_gemm_wide");
  } else {
    if (p.wm == 16) launch_ksplit<16>(stream, ta, tb, a, grid);
    else if (p.wm == 2) launch_ksplit<2>(stream, ta, tb, a, grid);
    else launch_ksplit<8>(stream, ta, tb, a, grid);
    check_launch("k_gemm_ksplit");
  }
  if (p.splits > 1) {
    const int64_t total = M * N;
    // from 65536 elements one thread each fills the chip
    if (total >= 65536)
      hipLaunchKernelGGL(k_splitk_sum, dim3((unsigned)cdiv(total, 256)), dim3(256), 0, stream, a.partial, p.splits, M,
                         total, out);
    else
      hipLaunchKernelGGL(k_splitk_reduce, dim3((unsigned)cdiv(total, 32)), dim3(256), 0, stream, a.partial, p.splits, M,
                         total, out);
    check_launch("k_splitk_reduce");
  }
}

void gemm_f64(hipStream_t stream, char transA, char transB, int64_t M, int64_t N, int64_t K,
              double alpha, const double* A, int64_t lda, const double* B, int64_t ldb,
              double beta, double* C, int64_t ldc, GemmWorkspace* ws) {
  GemmOut o;
  o.C1 = C; o.ldc1 = ldc; o.alpha1 = alpha; o.beta1 = beta; o.nsplit = N;
  o.C2 = C; o.ldc2 = ldc;
  gemm_f64(stream, transA, transB, M, N, K, A, lda, B, ldb, o, ws);
}

}  // namespace skema
