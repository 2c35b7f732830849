// MFMA GEMM C[m][n] = alpha * sum_k A[m][k] * B[n][k] with complex A (c128) and a real B whose rows are
// zero-padded to a multiple of 16 (ldb): the Cholesky contractions of a step whose vectors are real
// (vHS, Real3IndexFactorization.hpp:297-313) or whose trial is (vbias, 350-361).
//
// A 256-thread workgroup owns a TM x TN tile of C, each wavefront TM/2 x TN/2 of it; a k slice (16
// values, 8 for 128-row FP64 tiles) of A and B goes through LDS, double-buffered with one barrier per slice, in
// 16-byte pieces: consecutive lanes load consecutive pieces of a row. Rows in LDS are padded to an odd
// multiple of 16 bytes, so that the 16 rows of a fragment fall into different banks. FP32 converts A
// when it is staged. Along a 16-wide chunk lane group g takes k = k0 + 4 g + s in step s (FP32), the
// order of k_gemm_nt: both kernels give the same bits for the same split of k.
//
// Bound: MFMA. 128-row tiles take 10 LDS reads for 64 FP32 or 32 FP64 MFMAs (2048 matrix cycles) per
// slice and wavefront; the 64 x 64 tiles of k_gemm_nt 8-byte reads of single elements for half as
// many MFMAs, and twice the loads of B. Per launch, with the triangle of a symmetric vHS and the real
// vectors of a real trial against k_gemm_nt on the full ones (M 128, N 32, K 640, 1024 walkers):
// vHS FP64 905 -> 484 us, FP32 660 -> 288 us (128 x 128 tiles by the rule below; 247 with the 64 x 64
// that afq_autotune takes); vbias FP64 475 -> 230 us, FP32 277 -> 140 us. M 64,
// N 16, K 320, 512 walkers, FP64: vHS 68 -> 46 us.
//
// The compiler keeps the prefetched pieces of B (pb) of the 64- and 32-row FP64 tiles and of the 64 x 128
// FP32 ones in scratch, 48 bytes per lane: their loads are waited for before the MFMAs that they should
// run under, and vHS at M 128 writes 307 MB for 135 MB of V. The rates above and the plans below, fitted
// to measured times, contain that.
//
// The exchange as a quadratic form: sum_n tr(T_n^2) with T_n = G Lnak_n^T is G B G^T over the pairs
// (electron, orbital), B[(b, j)][(a, i)] = sum_n Lnak[n][b][i] Lnak[n][a][j] from the set-up. B is
// symmetric: 2 (N M)^2 flops per walker instead of the 4 N^2 M K of the T_n, and with K some multiples
// of M several times fewer, FP64 in place of the int8 split too. The Coulomb traces tr(T_n) are one
// more product with the flat Lnak rows. Exchange and traces, per Cholesky vector -> pair table:
//   M 128, N 32, K 640, 1024 walkers: FP64 6500, int8 2560 -> 790 + 230 us
//   M 64, N 16, K 320, 512 walkers: int8 166 -> 38 + 23 us
//   M 88, N 22, K 440, 137 walkers: int8 240 -> 42 + 27 us
//   M 77, N 19, K 385, 201 walkers, complex trial: FP64 490 -> 59 + 44 us
#include "afq_internal.hpp"

#include <algorithm>
#include <cmath>

namespace afq {

namespace {

constexpr int kXcds = 8;   // workgroups are dealt to them in turn

// DOT: the quadratic form A B A^T of each row instead of C, B being n x n and upper triangular (row q
// holds the entries p <= q). A workgroup takes an item, columns of tile_n times one chunk of the
// k <= its last column, and rows of a tile; it writes sum_q (A B)[row][q] A[row][q] over its share as
// that partial of the row (C[row][ldc]). kchunk is a multiple of TN.
// z = 1: the imaginary part of B, which follows the real part; its partials follow, times i.
template <typename R, int TM, int TN, int KS, bool DOT = false>
__global__ __launch_bounds__(256, 2) void k_gemm_real(int m, int n, int k, int kchunk, double alpha,
                                                      const double* __restrict__ A, long lda,
                                                      const R* __restrict__ B, long ldb,
                                                      double* __restrict__ C, long ldc,
                                                      long split_stride, int nanmix) {
  typedef typename acc_of<R>::type acc_t;
  constexpr bool F = sizeof(R) == 4;
  constexpr int SPS = KS / 4;                    // MFMA k steps of a slice
  constexpr int RA = KS * 2 * sizeof(R) + 16;    // staged row of A: an odd multiple of 16 bytes
  constexpr int RB = KS * sizeof(R) + 16;        // staged row of B
  static_assert(!F || KS == 16, "the FP32 sums keep 16-wide chunks");
  constexpr int MT = TM / 32, NT = TN / 32;      // 16-wide tiles of a wavefront
  constexpr int PA = TM * KS / 256;              // elements of A per thread and slice
  constexpr int BP = KS * (int)sizeof(R) / 16;   // 16-byte pieces of a row of B
  constexpr int PB = (TN * BP + 255) / 256;      // ... per thread and slice
  __shared__ __attribute__((aligned(16))) char sA[2][TM * RA];
  __shared__ __attribute__((aligned(16))) char sB[2][TN * RB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, r16 = lane & 15;
  const int wm = (wave >> 1) * (TM / 2), wn = (wave & 1) * (TN / 2);
  // column tiles fastest: consecutive workgroups (dealt round-robin to the XCDs) share rows of A,
  // and each XCD's L2 holds an eighth of B
  int tile_n = blockIdx.x, tile_m = blockIdx.y, kbeg = DOT ? 0 : blockIdx.z * kchunk, item = 0;
  if (DOT) {
    // each XCD takes a contiguous range of (tile_m, item), and the items of a chunk, one per tile_n from
    // the chunk's first column on, follow one another: its L2 holds the rows of A that they share
    const int nitem = gridDim.x, total = nitem * gridDim.y, b = blockIdx.x + nitem * blockIdx.y;
    const int q = total / kXcds, r = total % kXcds, xcd = b % kXcds;
    const int at = xcd * q + min(xcd, r) + b / kXcds;
    tile_m = at / nitem;
    item = at - tile_m * nitem;
    const int c = kchunk / TN;
    int x = item, len = (n + TN - 1) / TN;
    for (; x >= len; len -= c, kbeg += kchunk) x -= len;
    tile_n = kbeg / TN + x;
    B += blockIdx.z * (long)n * ldb;
  }
  const int kend = min(DOT ? min(k, (tile_n + 1) * TN) : k, kbeg + kchunk);
  if (!DOT) C += blockIdx.z * split_stride;

  double2 pa[PA];
  uint4 pb[PB];
  auto gload = [&](int k0) {
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      const int e = tid + 256 * i, row = e / KS, q = e % KS;
      const int gm = tile_m * TM + row;
      pa[i] = double2{0.0, 0.0};
      if (gm < m && k0 + q < kend)
        pa[i] = *reinterpret_cast<const double2*>(A + 2 * ((long)gm * lda + k0 + q));
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const int e = tid + 256 * i, row = e / BP, q = e % BP;
      const int gn = min(tile_n * TN + row, n - 1);
      if (PB * 256 == TN * BP || row < TN)
        pb[i] = *reinterpret_cast<const uint4*>(B + (long)gn * ldb + k0 + q * (16 / (int)sizeof(R)));
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      const int e = tid + 256 * i, row = e / KS, q = e % KS;
      R re = (R)pa[i].x, im = (R)pa[i].y;
      if (nanmix) {   // the zero imaginary part of B in a complex product: Inf or NaN spreads
        const R bad = (re - re) + (im - im);
        re += bad;
        im += bad;
      }
      R* p = reinterpret_cast<R*>(sA[buf] + row * RA) + 2 * q;
      p[0] = re;
      p[1] = im;
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const int e = tid + 256 * i, row = e / BP, q = e % BP;
      if (PB * 256 == TN * BP || row < TN)
        *reinterpret_cast<uint4*>(sB[buf] + row * RB + 16 * q) = pb[i];
    }
  };

  acc_t cr[MT][NT], ci[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) {
      cr[a][b] = acc_t{0, 0, 0, 0};
      ci[a][b] = acc_t{0, 0, 0, 0};
    }
  if (kbeg < kend) {
    gload(kbeg);
    sstore(0);
  }
  __syncthreads();
  for (int k0 = kbeg, buf = 0; k0 < kend; k0 += KS, buf ^= 1) {
    const bool more = k0 + KS < kend;
    if (more) gload(k0 + KS);
    R ar[MT][SPS], ai[MT][SPS], br[NT][SPS];
    // lane group g: steps s = 0 .. SPS - 1 at k0 + SPS g + s, contiguous in its row
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const char* p = sA[buf] + (wm + 16 * t + r16) * RA + g * SPS * 2 * (int)sizeof(R);
#pragma unroll
      for (int h = 0; h < (F ? SPS / 2 : SPS); ++h) {
        if constexpr (F) {
          const float4 x = reinterpret_cast<const float4*>(p)[h];
          ar[t][2 * h] = x.x;
          ai[t][2 * h] = x.y;
          ar[t][2 * h + 1] = x.z;
          ai[t][2 * h + 1] = x.w;
        } else {
          const double2 x = reinterpret_cast<const double2*>(p)[h];
          ar[t][h] = x.x;
          ai[t][h] = x.y;
        }
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const char* p = sB[buf] + (wn + 16 * t + r16) * RB + g * SPS * (int)sizeof(R);
      if constexpr (F) {
        const float4 x = *reinterpret_cast<const float4*>(p);
        br[t][0] = x.x;
        br[t][1] = x.y;
        br[t][2] = x.z;
        br[t][3] = x.w;
      } else {
#pragma unroll
        for (int h = 0; h < SPS / 2; ++h) {
          const double2 x = reinterpret_cast<const double2*>(p)[h];
          br[t][2 * h] = x.x;
          br[t][2 * h + 1] = x.y;
        }
      }
    }
#pragma unroll
    for (int s = 0; s < SPS; ++s)
#pragma unroll
      for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b) {
          cr[a][b] = mfma16x16x4(ar[a][s], br[b][s], cr[a][b]);
          ci[a][b] = mfma16x16x4(ai[a][s], br[b][s], ci[a][b]);
        }
    // the other buffer was last read in the previous slice, before the barrier that ended it
    if (more) sstore(buf ^ 1);
    __syncthreads();
  }
  if constexpr (DOT) {
    double2* red = reinterpret_cast<double2*>(sA);   // [2][TM], after the last barrier of the loop
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = wm + 16 * a + acc_row<R>(g, r), gm = min(tile_m * TM + row, m - 1);
        double er = 0.0, ei = 0.0;
#pragma unroll
        for (int b = 0; b < NT; ++b) {
          const int col = tile_n * TN + wn + 16 * b + r16;
          if (col < n) {
            const double2 x = *reinterpret_cast<const double2*>(A + 2 * ((long)gm * lda + col));
            er += cr[a][b][r] * x.x - ci[a][b][r] * x.y;
            ei += cr[a][b][r] * x.y + ci[a][b][r] * x.x;
          }
        }
        er = row_sum16(er);
        ei = row_sum16(ei);
        if (r16 == 15) red[(wave & 1) * TM + row] = double2{er, ei};
      }
    __syncthreads();
    if (tid < TM && tile_m * TM + tid < m) {
      const double2 x = red[tid], y = red[TM + tid];
      const double re = x.x + y.x, im = x.y + y.y;
      *reinterpret_cast<double2*>(
          C + 2 * ((long)(tile_m * TM + tid) * ldc + blockIdx.z * gridDim.x + item)) =
          blockIdx.z ? double2{-im, re} : double2{re, im};
    }
    return;
  }
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) {
      const int col = tile_n * TN + wn + 16 * b + r16;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = tile_m * TM + wm + 16 * a + acc_row<R>(g, r);
        if (row < m && col < n) {
          const double2 v = double2{alpha * (double)cr[a][b][r], alpha * (double)ci[a][b][r]};
          *reinterpret_cast<double2*>(C + 2 * ((long)row * ldc + col)) = v;
        }
      }
    }
}

// Bp[row][0..ldb) = src[r(row)][0..k), zero-padded; packed: row p of the upper triangle i <= j of an
// n x n set of rows is source row i n + j
template <typename D>
__global__ void k_pad_rows(long rows, int k, int ldb, int n, int packed,
                           const double* __restrict__ src, int stride, D* __restrict__ dst) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= rows * ldb) return;
  const long p = e / ldb;
  const int c = (int)(e - p * ldb);
  long r = p;
  if (packed) {
    // i: largest with i (2 n - i + 1) / 2 <= p
    int i = (int)((2.0 * n + 1.0 - sqrt((2.0 * n + 1.0) * (2.0 * n + 1.0) - 8.0 * (double)p)) * 0.5);
    i = max(0, min(i, n - 1));
    while ((long)i * (2 * n - i + 1) / 2 > p) --i;
    while (i + 1 < n && (long)(i + 1) * (2 * n - i) / 2 <= p) ++i;
    r = (long)i * n + i + (p - (long)i * (2 * n - i + 1) / 2);
  }
  dst[e] = c < k ? (D)src[(r * k + c) * stride] : (D)0;
}

// B[q = (b, j)][p = (a, i)] = w sum_n L[n][a][j] L[n][b][i], w = 2 for p < q, 1 for p = q and 0 above:
// the product D^T D of D[n][(a, j)] with the second indices of its rows and columns exchanged. Each
// wavefront computes 64 x 64 of it from L in L2 (set-up only: 0.4 ms at N M = 4096, 640 vectors).
// LC: complex L, block z = 0 the real and z = 1 the imaginary part of B.
template <bool LC>
__global__ __launch_bounds__(256, 2) void k_pair_table(int M, int NM, int K, const double* __restrict__ L,
                                                       long ldl, double* __restrict__ B, long ldb) {
  const bool imag = LC && blockIdx.z == 1;
  B += blockIdx.z * (long)NM * ldb;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, r16 = lane & 15;
  const int r0 = blockIdx.y * 128 + (wave >> 1) * 64, s0 = blockIdx.x * 128 + (wave & 1) * 64;
  d4 acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = d4{0, 0, 0, 0};
  for (int n0 = 0; n0 < K; n0 += 4) {
    const int n = n0 + g;
    const double* row = L + (long)min(n, K - 1) * ldl;
    double x[4], y[4], x2[4], y2[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int rr = min(r0 + 16 * t + r16, NM - 1), sc = min(s0 + 16 * t + r16, NM - 1);
      if (LC) {
        const double2 xc = reinterpret_cast<const double2*>(row)[rr];
        const double2 yc = reinterpret_cast<const double2*>(row)[sc];
        x[t] = xc.x;
        x2[t] = imag ? xc.y : -xc.y;
        y[t] = imag ? yc.y : yc.x;
        y2[t] = imag ? yc.x : yc.y;
      } else {
        x[t] = row[rr];
        y[t] = row[sc];
        x2[t] = 0.0;
      }
      if (n >= K) x[t] = x2[t] = 0.0;
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        acc[a][b] = mfma16x16x4(x[a], y[b], acc[a][b]);
        if (LC) acc[a][b] = mfma16x16x4(x2[a], y2[b], acc[a][b]);
      }
  }
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int sc = s0 + 16 * b + r16, eb = sc / M, i = sc - eb * M;
    if (sc >= NM) continue;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int rr = r0 + 16 * a + acc_row<double>(g, r);
        if (rr >= NM) continue;
        const int ea = rr / M, j = rr - ea * M, q = eb * M + j, p = ea * M + i;
        B[(long)q * ldb + p] = p < q ? 2.0 * acc[a][b][r] : (p == q ? acc[a][b][r] : 0.0);
      }
  }
}

// Rows of a tile, chunk of k and partials per row and table of the quadratic form (columns in tiles of
// 64). The chunk is the smallest from 128 on with at most max_parts partials and 64 workgroups per CU.
// The tile is the largest unless a smaller one has 5 % less estimated time: rounds of the 2, 3 or 4
// workgroups that a CU holds, a last one alone counting 1.6, times the rows (0.9 of the rate for 32).
// 128, 64 and 32 rows take 48, 38 and 39 us at M 64, N 16 with 512 walkers; 64 and 32 rows 42 and 45
// at M 88, N 22 with 137, and 70 and 59 at M 77, N 19 with 201 and two tables.
struct PairPlan {
  int tm, chunk, parts;
  double cost;   // rounds times rows times the mean k of an item
};
PairPlan pair_plan(int W, int NM, int planes, int max_parts) {
  const int nt = (NM + 63) / 64, cus = device_cus();
  PairPlan best{};
  double best_cost = 0.0;
  for (int tm = 128, held = 2; tm >= 32; tm /= 2, ++held) {
    const long rows = (W + tm - 1) / tm;
    PairPlan p;
    p.tm = tm;
    for (p.chunk = 128;; p.chunk *= 2) {
      const int c = p.chunk / 64;
      p.parts = 0;
      for (int t = 0; t < nt; ++t) p.parts += t / c + 1;
      if (c >= nt || (p.parts <= max_parts / planes && p.parts * rows <= 64L * cus)) break;
    }
    const long n = (p.parts * rows * planes + cus - 1) / cus, r = n % held;
    const double rounds = (n - r + (r > 0 ? std::max((double)r, 1.6) : 0.0)) / (tm == 32 ? 0.9 : 1.0);
    const double cost = rounds * tm * p.chunk;
    if (tm == 128 || cost < 0.95 * best_cost) {
      p.cost = rounds * tm * 32.0 * nt * (nt + 1) / p.parts;
      best = p;
      best_cost = cost;
    }
  }
  return best;
}

// FP64: the tile and the split of k with the shortest estimated time: workgroups of the fullest CU times
// the work of one (234 GFLOP/s per CU, 0.234e6 FLOP per us, where workgroups share it, 0.6 of it for one alone; the
// smaller tiles at 0.95 and 0.8 of that), and the pass that adds the splits. Returns that time in us.
double gemm_f64_plan(int m, int n, int k, long split_elems, int& tm, int& tn, int& splits) {
  const double cus = device_cus();
  double best = 1e300;
  const int tiles[3][2] = {{128, 64}, {64, 64}, {64, 32}};
  const double eff[3] = {1.0, 0.95, 0.8};
  for (int t = 0; t < 3; ++t)
    for (int s = 1; s <= kMaxSplits; ++s) {
      if (s > 1 && (k / s < 128 || (long)s * m * n > split_elems)) break;
      const double wgs = std::ceil((double)m / tiles[t][0]) * std::ceil((double)n / tiles[t][1]) * s;
      const double share = std::ceil(wgs / cus);
      double us = share * 4.0 * tiles[t][0] * tiles[t][1] * std::ceil((double)k / s) / (0.234e6 * eff[t]);
      if (share < 2) us /= 0.6;
      if (s > 1) us += 4.0 + 16e-6 * m * (double)n * (s + 1) / 4.0;
      if (us < 0.98 * best) {
        best = us;
        tm = tiles[t][0];
        tn = tiles[t][1];
        splits = s;
      }
    }
  return best;
}

}  // namespace

size_t pair_table_elems(int NM, bool real) { return (real ? 1 : 2) * (size_t)NM * gemm_real_row(NM); }

void launch_pair_table(hipStream_t s, int M, int N, int K, const double* L, bool real, double* B) {
  const int NM = N * M, nt = (NM + 127) / 128;
  const long ldb = gemm_real_row(NM);
  AFQ_HIP(hipMemsetAsync(B, 0, pair_table_elems(NM, real) * sizeof(double), s));   // the rows' padding
  if (real)
    hipLaunchKernelGGL(k_pair_table<false>, dim3(nt, nt), dim3(256), 0, s, M, NM, K, L, ldb, B, ldb);
  else
    hipLaunchKernelGGL(k_pair_table<true>, dim3(nt, nt, 2), dim3(256), 0, s, M, NM, K, L, 2L * NM, B, ldb);
  AFQ_HIP(hipGetLastError());
}

int pair_parts(int W, int NM, bool real, int max_parts) {
  const int planes = real ? 1 : 2;
  return planes * pair_plan(W, NM, planes, max_parts).parts;
}

double pair_exchange_cost(int W, int NM, bool real, int max_parts) {
  return pair_plan(W, NM, real ? 1 : 2, max_parts).cost;
}

double gemm_f64_us(int m, int n, int k, long split_elems) {
  int tm, tn, splits;
  return gemm_f64_plan(m, n, k, split_elems, tm, tn, splits);
}

void launch_pair_exchange(hipStream_t s, int W, int NM, bool real, int max_parts, const double* G,
                          const double* B, double* part) {
  if (W <= 0) return;
  const int planes = real ? 1 : 2;
  const PairPlan p = pair_plan(W, NM, planes, max_parts);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(p.parts, (W + p.tm - 1) / p.tm, planes), dim3(256), 0, s, W, NM, NM, p.chunk,
                       1.0, G, (long)NM, B, (long)gemm_real_row(NM), part, (long)planes * p.parts, 0L, 1);
  };
  if (p.tm == 128) go(k_gemm_real<double, 128, 64, 8, true>);
  else if (p.tm == 64) go(k_gemm_real<double, 64, 64, 16, true>);
  else go(k_gemm_real<double, 32, 64, 16, true>);
  AFQ_HIP(hipGetLastError());
}

// FP64 takes the tile of gemm_f64_plan
int gemm_real_tile_configs(int precision) { return precision == AFQ_FP64 ? 1 : 4; }

int gemm_real_row(int k) { return (k + 15) / 16 * 16; }

void launch_pad_rows(hipStream_t s, long rows, int k, int packed_n, const double* src, bool complex_src,
                     double* dst) {
  const int ldb = gemm_real_row(k);
  hipLaunchKernelGGL(k_pad_rows<double>, dim3((unsigned)((rows * ldb + 255) / 256)), dim3(256), 0, s,
                     rows, k, ldb, packed_n, packed_n > 0 ? 1 : 0, src, complex_src ? 2 : 1, dst);
  AFQ_HIP(hipGetLastError());
}

void launch_pad_rows(hipStream_t s, long rows, int k, int packed_n, const double* src, bool complex_src,
                     float* dst) {
  const int ldb = gemm_real_row(k);
  hipLaunchKernelGGL(k_pad_rows<float>, dim3((unsigned)((rows * ldb + 255) / 256)), dim3(256), 0, s,
                     rows, k, ldb, packed_n, packed_n > 0 ? 1 : 0, src, complex_src ? 2 : 1, dst);
  AFQ_HIP(hipGetLastError());
}

void launch_gemm_real(hipStream_t s, int precision, int m, int n, int k, double alpha,
                      const double* A, long lda, const void* B, double* C, long ldc, bool nanmix,
                      double* split_ws, long split_ws_elems, int cfg) {
  if (m <= 0 || n <= 0) return;
  const bool f32 = precision != AFQ_FP64;
  // the splits of launch_gemm_nt_z: the FP32 sums keep their order
  int splits = split_ws ? gemm_splits(m, n, k) : 1;
  if ((long)splits * m * n > split_ws_elems) splits = 1;
  int tm = 64, tn = 32;
  if (!f32) gemm_f64_plan(m, n, k, split_ws ? split_ws_elems : 0, tm, tn, splits);
  int kchunk = (k + splits - 1) / splits;
  kchunk = (kchunk + 31) & ~31;
  splits = std::max(1, (k + kchunk - 1) / kchunk);
  // FP32: the largest tile that still gives two workgroups per CU (128 x 128: four, so that a partly
  // filled last round costs little), else 64 x 32: 512 walkers of 64 orbitals are 264 64 x 64 tiles
  // of vHS, one workgroup on most CUs with every load exposed.
  // cfg (FP32; 0: this rule) bit 0: the other row count, bit 1: the other column count.
  if (f32) {
    const long cus = device_cus();
    auto tiles = [&](int a, int b) { return (long)((m + a - 1) / a) * ((n + b - 1) / b) * splits; };
    if (tiles(128, 128) >= 4 * cus) tm = tn = 128;
    else if (tiles(128, 64) >= 2 * cus) tm = 128, tn = 64;
    else if (tiles(64, 64) >= 2 * cus) tn = 64;
  }
  if (f32 && (cfg & 1)) tm = tm == 64 ? 128 : 64;
  if (f32 && (cfg & 2)) tn = tn == 64 ? 128 : 64;
  if (tm == 128 && tn == 32) tn = 64;
  const dim3 grid((n + tn - 1) / tn, (m + tm - 1) / tm, splits);
  double* out = splits > 1 ? split_ws : C;
  const long ldo = splits > 1 ? n : ldc;
  const long sstride = splits > 1 ? 2L * m * n : 0;
  const double a = splits > 1 ? 1.0 : alpha;
  const long ldb = gemm_real_row(k);
  auto go = [&](auto kern, auto* b) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, m, n, k, kchunk, a, A, lda, b, ldb, out, ldo,
                       sstride, nanmix ? 1 : 0);
  };
  if (f32) {
    const float* b = (const float*)B;
    if (tm == 128) tn == 128 ? go(k_gemm_real<float, 128, 128, 16>, b) : go(k_gemm_real<float, 128, 64, 16>, b);
    else if (tn == 128) go(k_gemm_real<float, 64, 128, 16>, b);
    else tn == 64 ? go(k_gemm_real<float, 64, 64, 16>, b) : go(k_gemm_real<float, 64, 32, 16>, b);
  } else {
    const double* b = (const double*)B;
    if (tm == 128) go(k_gemm_real<double, 128, 64, 8>, b);
    else tn == 64 ? go(k_gemm_real<double, 64, 64, 16>, b) : go(k_gemm_real<double, 64, 32, 16>, b);
  }
  AFQ_HIP(hipGetLastError());
  if (splits > 1) launch_split_reduce(s, m, n, splits, alpha, split_ws, C, ldc);
}

}  // namespace afq
