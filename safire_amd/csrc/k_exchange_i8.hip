// Exchange and Coulomb energy (Real3IndexFactorization::energy_impl, Real3IndexFactorization.hpp:
// 476-559) with the contraction T_wn = G_w Lnak_n^T on int8 MFMA (v_mfma_i32_16x16x64_i8),
// split after Ozaki: every row of G and of each Lnak_n is scaled by a power of two u and
// written as a sum of int8 slices, x = u (q0 + q1/254 + q2/254^2 + ...) with every |qs| <= 127
// (q0 = rint(x/u), |x/u| < 127; each residual lies in [-1/2, 1/2], times 254 in [-127, 127]).
// A slice product accumulates in int32 without rounding, so the error left is the truncation
// of the slice series, relative to the row maximum.
//
// Slices: 6 of G and 6 of each Lnak row, and per Cholesky vector a slice-product order o_n in 2..5 (4 or
// 5 for up to 16 electrons: every T then to 254^-5 of its own vector's size, whatever the sizes of the
// others) with all products s + t <= o_n kept (21, 15, 10 or 6), fixed at set-up from the vector's size
// r_n = max|L_n| / max_m |L_m|: o_n = ceil(5 + 2 log_254 r_n). The error a vector adds to EXX
// scales as r_n^2 254^-(o_n + 1) (both its T block and the truncation of its product series are
// proportional to r_n), so every vector then contributes at most 254^-6 of the largest one's
// scale: on Cholesky vectors whose sizes decay, the large vectors take all 21 products and the
// small ones few, fewer products on average than a uniform order 4 (15) for tens of times less
// error. The truncation of G is the same for every Cholesky vector and adds up coherently.
//
// Structure: one product of the flat row sets (w, b) and (n, a). A workgroup takes Rw walkers
// (Rw N <= 16 NW rows) and per pass Cv vectors (Cv N <= 16 CT columns), so the 16-wide tiles are
// filled across walkers and vectors (22 electrons: 110 of 128 rows and 44 of 48 columns, where
// padding to 32 x 32 blocks uses 47 %). Each wavefront slices its 16 rows of G once into A
// fragments that stay in registers. The slices of a pass's columns are loaded into registers while
// the previous pass is multiplied, and stored to LDS between two barriers; only the slices that
// the pass's order needs are loaded. Real trial orbitals give Im Lnak = 0: only real slices are
// kept then (LC = false), with 2 MFMAs per slice product instead of 4.
// T = uG_a uL_b sum_o 254^-o acc_o is assembled in FP64 (orders that fit are joined exactly in int32
// first) and goes to LDS, where the next pass forms tr(T^2) and tr(T): two T buffers when they fit,
// and then half of the wavefronts do that before their MFMAs and half after, so that the VALU work
// of one wavefront of a SIMD runs under the MFMAs of the other.
//
// What bounds it: neither unit alone. A pass is MFMAs (8 K of 12 K cycles at M = 128), pair sums and
// the two barriers around the LDS store, and the two wavefronts of a SIMD go through them nearly
// together. One walker's 32 x 32 blocks with complex slices against this for real trials: M 128, N 32,
// K 640, W 1024: 4040 -> 2560 us; M 88, N 22, K 440, W 137: 1055 -> 240 us. Where padding costs less than
// that, and in small calls, k_exchange_i8w.hip is taken (per_walker below), and with enough vectors and
// walkers the quadratic form over the pair table in FP64 (k_gemm_real.hip: 1020 and 69 us for these,
// traces included).
//
// M <= 128, N <= 32.
#include "i8_split.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace afq {

namespace {

using namespace i8;

constexpr int kMaxKC = 2;         // 64-wide k chunks: M <= 128
constexpr int kItems = 8;         // pairs of a pass per thread, at most

template <int KC, int CT, bool LC, int NW>
__global__ __launch_bounds__(64 * NW, NW / 4) void k_exchange_i8(
    int W, int M, int N, int K, int Mp, int Rw, int Cv, int chunk, int tdbl,
    const double* __restrict__ G, const int8_t* __restrict__ Lq, const double* __restrict__ Lu,
    const int* __restrict__ ord, double* __restrict__ Kl, double* __restrict__ part, int nchunk) {
  constexpr int kThreads = 64 * NW;
  constexpr int NP = LC ? 2 : 1;                 // real and imaginary planes of a slice
  constexpr int PCS = (kS * NP * 16 * CT * 4 * KC + kThreads - 1) / kThreads;   // 16-byte pieces per thread
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int crows = Cv * N;                      // staged columns
  const int ldt = (crows + 1) & ~1;              // row of T: ldt + 1 odd, distinct banks down a diagonal
  const int rowb = 16 * ((Mp >> 4) | 1);         // staged row: odd multiple of 16 bytes
  const int planeb = crows * rowb;
  const int tsize = 16 * NW * ldt;
  double2* sT = reinterpret_cast<double2*>(smem);                        // [1 or 2][16 NW][ldt]
  double* sU = reinterpret_cast<double*>(sT + (tdbl ? 2 : 1) * tsize);   // [16 CT] column units
  int* sO = reinterpret_cast<int*>(sU + 16 * CT);                        // order of the next pass
  double* sR = reinterpret_cast<double*>(sO + 4);                        // [16 NW] row units / 254
  char* sB = reinterpret_cast<char*>(sR + 16 * NW);                          // [slice][plane][crows][rowb]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int w0 = blockIdx.x * Rw;
  const int nw = min(Rw, W - w0);
  const int nbeg = blockIdx.y * chunk, nend = min(K, nbeg + chunk);
  const size_t plane = (size_t)K * N * Mp;       // bytes of one slice plane

  // ---- slices of the wavefront's rows of G: row 16 wave + r16, k = 64 kc + 16 g + j (j < 16)
  i4 ar[KC][kS], ai[KC][kS];
  const int grow = 16 * wave + r16;
  const bool gok = grow < nw * N;
  const double uG = slice_row<KC>(reinterpret_cast<const double2*>(G) + ((long)w0 * N + (gok ? grow : 0)) * M, gok,
                                  M, g, ar, ai);
  // units of the rows, over 254: the joined orders 0 and 1 carry one factor 254
  if (lane < 16) sR[16 * wave + lane] = uG * (1.0 / kBase);

  // ---- staging: the rows of a plane are contiguous, so a pass is crows Mp bytes of each plane
  const int per = crows * (Mp >> 4);             // pieces of a plane
  unsigned piece[PCS];                           // plane << 20 | byte in sB
#pragma unroll
  for (int i = 0; i < PCS; ++i) {
    const int q = tid + i * kThreads;
    const int pl = q / per, o = q - pl * per;
    const int row = o / (Mp >> 4), kv = o - row * (Mp >> 4);
    piece[i] = (unsigned)pl << 20 | (unsigned)(pl * planeb + row * rowb + 16 * kv);
  }
  uint4 pre[PCS];
  double preU = 0.0;
  int preO = 2;
  // the slices and units of the pass at n0, and the orders of the vectors of the pass after it
  auto gload = [&](int n0, int on) {
    const size_t first = (size_t)n0 * N * Mp;
#pragma unroll
    for (int i = 0; i < PCS; ++i) {
      pre[i] = uint4{0u, 0u, 0u, 0u};
      const int pl = piece[i] >> 20;
      const size_t off = first + 16u * (unsigned)(tid + i * kThreads - pl * per);
      if (pl < (on + 1) * NP && off < plane)
        pre[i] = *reinterpret_cast<const uint4*>(Lq + pl * plane + off);
    }
    const long col = (long)n0 * N + tid;
    if (tid < crows) preU = col < (long)K * N ? Lu[col] : 0.0;
    if (tid < Cv) preO = n0 + Cv + tid < nend ? ord[n0 + Cv + tid] : 2;
  };
  auto lstore = [&](int on) {
#pragma unroll
    for (int i = 0; i < PCS; ++i)
      if ((int)(piece[i] >> 20) < (on + 1) * NP)
        *reinterpret_cast<uint4*>(sB + (piece[i] & 0xfffff)) = pre[i];
    if (tid < crows) sU[tid] = preU;
    if (wave == 0) {   // Cv <= 48 vectors
      int o = preO;
      for (int off = 32; off > 0; off >>= 1) o = max(o, __shfl_xor(o, off, 64));
      if (tid == 0) sO[0] = o;
    }
  };

  // ---- pairs of a pass: thread t of a walker takes (a, a + d mod N) of vector v for its items,
  // d = 0 .. N/2; together each unordered pair once (twice with half the weight when 2 d = N).
  // Packed element offsets x = (a, b), y = (b, a) into T (15 bits each), bits 30, 31: the weight.
  const int tpw = kThreads / Rw;
  const int wl = tid / tpw, tl = tid - wl * tpw;
  // A thread without a further item reads its walker's first element with weight 0.
  unsigned item[kItems];
  const int D = N / 2 + 1;
  const int nitem = (Cv * N * D + tpw - 1) / tpw;
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int q = tl + i * tpw;
    const int a = q % N, d = (q / N) % D, v = (q / N) / D;
    const int b = a + d >= N ? a + d - N : a + d;
    const unsigned x = (wl * N + a) * ldt + v * N + b, y = (wl * N + b) * ldt + v * N + a;
    item[i] = x | (y << 15) | ((d == 0 || 2 * d == N) ? 0x40000000u : 0x80000000u);
    if (wl >= nw) item[i] = 0;
    else if (v >= Cv) item[i] = (wl * N * ldt) | (wl * N * ldt) << 15;
  }
  const int gs = N <= 4 ? 4 : (N <= 8 ? 8 : 16);   // lanes per (walker, vector) trace
  double exx_re = 0.0, exx_im = 0.0;
  auto pairs = [&](const double2* T, int n0) {
    // vectors past K have T = 0 (their slices and units are staged as zero)
#pragma unroll
    for (int i = 0; i < kItems; i += 2) {
      if (i < nitem) {   // uniform
        const double2 x0 = T[item[i] & 0x7fff], y0 = T[(item[i] >> 15) & 0x7fff];
        const double2 x1 = T[item[i + 1] & 0x7fff], y1 = T[(item[i + 1] >> 15) & 0x7fff];
        const double w0_ = (double)(item[i] >> 30), w1_ = (double)(item[i + 1] >> 30);
        exx_re = fma(w0_, fma(-x0.y, y0.y, x0.x * y0.x), exx_re);
        exx_im = fma(w0_, fma(x0.x, y0.y, x0.y * y0.x), exx_im);
        exx_re = fma(w1_, fma(-x1.y, y1.y, x1.x * y1.x), exx_re);
        exx_im = fma(w1_, fma(x1.x, y1.y, x1.y * y1.x), exx_im);
      }
    }
    const int nv = min(Cv, nend - n0);
    const int np = nw * nv;
    // traces: consecutive (walker, vector) pairs go to different wavefronts
    for (int p0 = 0; p0 + wave < np; p0 += kThreads / gs) {
      const int p = p0 + wave + NW * (lane / gs);
      const int w = p / nv, v = p - w * nv;
      const bool in = p < np;
      const double2* Td = T + w * N * ldt + v * N;
      const int a = lane & (gs - 1);
      double2 x = double2{0.0, 0.0}, y = x;
      if (in && a < N) x = Td[a * (ldt + 1)];
      if (in && a + gs < N) y = Td[(a + gs) * (ldt + 1)];
      double dr = x.x + y.x, di = x.y + y.y;
      if (gs == 16) {
        dr = row_sum16(dr);
        di = row_sum16(di);
      } else {
        for (int off = 1; off < gs; off <<= 1) {
          const double ur = __shfl_up(dr, off, 64), ui = __shfl_up(di, off, 64);
          if (a >= off) {
            dr += ur;
            di += ui;
          }
        }
      }
      if (in && a == gs - 1)
        *reinterpret_cast<double2*>(Kl + 2 * ((long)(w0 + w) * K + n0 + v)) = double2{dr, di};
    }
  };

  // ---- one column tile with the slice products s + t <= ON: T rows of this wavefront to LDS
  auto tile = [&](auto on_c, int t, double2* T) {
    constexpr int ON = decltype(on_c)::value;
    i4 cR[ON + 1], cI[ON + 1], cQ[LC ? ON + 1 : 1];
#pragma unroll
    for (int o = 0; o <= ON; ++o) {
      cR[o] = i4{0, 0, 0, 0};
      cI[o] = i4{0, 0, 0, 0};
      if (LC) cQ[o] = i4{0, 0, 0, 0};
    }
    const int col = 16 * t + r16;
    // columns past the pass read its last row and are not stored; bytes past a row meet zeros of G
    int base = min(col, crows - 1) * rowb + 16 * g;
    // two chunks: one opaque address per tile, not those of all slices held over the tiles in
    // registers that are then spilled (M = 88, N = 22: 254 -> 240 us)
    if (KC > 1) asm volatile("" : "+v"(base));
#pragma unroll
    for (int kc = 0; kc < KC; ++kc)
#pragma unroll
      for (int q = 0; q <= ON; ++q) {
        const i4 br = *reinterpret_cast<const i4*>(sB + base + q * NP * planeb + 64 * kc);
        const i4 bi = LC ? *reinterpret_cast<const i4*>(sB + base + (q * NP + 1) * planeb + 64 * kc) : br;
#pragma unroll
        for (int s = 0; s + q <= ON; ++s) {
          cR[s + q] = mfma_i8(ar[kc][s], br, cR[s + q]);
          cI[s + q] = mfma_i8(ai[kc][s], br, cI[s + q]);
          if (LC) {
            cQ[LC ? s + q : 0] = mfma_i8(ai[kc][s], bi, cQ[LC ? s + q : 0]);
            cI[s + q] = mfma_i8(ar[kc][s], bi, cI[s + q]);
          }
        }
      }
    if (LC)
#pragma unroll
      for (int o = 0; o <= ON; ++o) cR[o] -= cQ[LC ? o : 0];
    const double uL = sU[min(col, crows - 1)];
    if (col < crows) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double u = sR[16 * wave + 4 * g + r] * uL;
        T[(16 * wave + 4 * g + r) * ldt + col] = double2{join_orders<ON, KC, LC>(cR, r) * u, join_orders<ON, KC, LC>(cI, r) * u};
      }
    }
  };

  int on = 2;
  if (nbeg < nend) {
    for (int n = nbeg; n < min(nbeg + Cv, nend); ++n) on = max(on, ord[n]);
    on = __builtin_amdgcn_readfirstlane(on);
    gload(nbeg, on);
    lstore(on);
  }
  __syncthreads();
  int tb = 0;
  for (int n0 = nbeg; n0 < nend; n0 += Cv) {
    const bool more = n0 + Cv < nend, prev = n0 > nbeg;
    const int next = __builtin_amdgcn_readfirstlane(sO[0]);
    if (more) gload(n0 + Cv, next);
    double2* T = sT + (tdbl ? tb * tsize : 0);
    const double2* Tp = sT + (tdbl ? (tb ^ 1) * tsize : 0);
    if (prev && (!tdbl || wave < NW / 2)) pairs(Tp, n0 - Cv);
    if (!tdbl) lds_barrier();   // the previous pass's T has been read
    for (int t = 0; t < CT; ++t) {
      if (on == 5) tile(std::integral_constant<int, 5>(), t, T);
      else if (on == 4) tile(std::integral_constant<int, 4>(), t, T);
      else if (on == 3) tile(std::integral_constant<int, 3>(), t, T);
      else tile(std::integral_constant<int, 2>(), t, T);
    }
    if (prev && tdbl && wave >= NW / 2) pairs(Tp, n0 - Cv);
    lds_barrier();              // this pass's slices have been read, its T is written
    if (more) lstore(next);
    lds_barrier();
    on = next;
    tb ^= 1;
  }
  if (nbeg < nend)
    pairs(sT + (tdbl ? (tb ^ 1) * tsize : 0), nbeg + (nend - 1 - nbeg) / Cv * Cv);

  // ---- per-walker sums of the threads' partials, in a fixed order: 8 threads per walker
  __syncthreads();
  sT[tid] = double2{exx_re, exx_im};
  __syncthreads();
  for (int w = tid >> 3; w < Rw; w += kThreads / 8) {
    double re = 0.0, im = 0.0;
    for (int t = tid & 7; t < tpw; t += 8) {
      const double2 x = sT[w * tpw + t];
      re += x.x;
      im += x.y;
    }
    for (int off = 4; off > 0; off >>= 1) {
      re += __shfl_xor(re, off, 8);
      im += __shfl_xor(im, off, 8);
    }
    if ((tid & 7) == 0 && w < nw)
      *reinterpret_cast<double2*>(part + 2 * ((long)(w0 + w) * nchunk + blockIdx.y)) =
          double2{re, im};
  }
}

// per Cholesky vector n: vmax[n] = max |component| of Lnak_n (one workgroup per vector)
__global__ void k_vector_max(long per, const double* __restrict__ L, double* __restrict__ vmax) {
  const long n = blockIdx.x;
  double m = 0.0;
  for (long e = threadIdx.x; e < 2 * per; e += blockDim.x) m = fmax(m, fabs(L[2 * n * per + e]));
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
  __shared__ double red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) vmax[n] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

// Lq[t][p][row][0..Mp) = slice t of part p (0: real, 1: imaginary, the latter only with np = 2)
// of row Lnak[n][b][:] / Lu[n][b] (zero for k >= M); one wavefront per row, lanes over k
__global__ __launch_bounds__(256) void k_split_lnak_i8(int rows, int M, int Mp, int np,
                                                       const double* __restrict__ L,
                                                       int8_t* __restrict__ Lq,
                                                       double* __restrict__ Lu) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= rows) return;
  const double* x = L + 2 * (long)row * M;
  double mx = 0.0;
  for (int k = lane; k < 2 * M; k += 64) mx = fabs(x[k]) <= 1.0e300 ? fmax(mx, fabs(x[k])) : INFINITY;
  for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
  bool zero;
  const double u = row_unit(mx, zero);
  const double inv = (u == u && !zero) ? 1.0 / u : 0.0;
  if (lane == 0) Lu[row] = u;
  const size_t plane = (size_t)rows * Mp;
  for (int k = lane; k < Mp; k += 64)
    for (int p = 0; p < np; ++p) {
      int q[kS];
      slice(k < M && inv != 0.0 ? x[2 * k + p] * inv : 0.0, q);
#pragma unroll
      for (int t = 0; t < kS; ++t) Lq[(t * np + p) * plane + (size_t)row * Mp + k] = (int8_t)q[t];
    }
}

struct Plan {
  int nw, ct, rw, cv, chunk, nchunk, tdbl;
  size_t lds;
};

constexpr size_t kLdsMax = 160 * 1024;

size_t lds_of(int nw, int ct, int cv, int N, int Mp, int np, int tdbl) {
  const int crows = cv * N, ldt = (crows + 1) & ~1;
  // T, column units, slices, and the reads past the last staged row
  return sizeof(double2) * (size_t)(tdbl ? 2 : 1) * 16 * nw * ldt + 8 * (size_t)16 * (ct + nw) + 16 +
         (size_t)kS * np * crows * 16 * ((Mp >> 4) | 1) + 128;
}

// Column tiles: 2 (32 columns) or, where it packs the vectors better, 3; T is double-buffered
// where LDS allows (worth 15 %, the pair sums then overlap the MFMAs). 8 wavefronts (two per
// SIMD), or 4 where workgroups of 8 would leave CUs without work. The vectors are split into
// chunks that minimise the rounds of workgroups times (passes + 2), the 2 standing for reading and
// slicing the workgroup's G.
Plan tiles_of(int W, int M, int N, int K, int np, double* eff) {
  const int Mp = exchange_i8_row(M);
  const long cus = device_cus();
  Plan p{};
  double best = -1.0;
  auto shape = [&](int nw) {
    best = -1.0;
    for (int ct = 2; ct <= 3; ++ct) {
      const int cv = std::min(16 * ct / N, K);
      if (cv < 1) continue;
      for (int td = 1; td >= 0; --td) {
        const size_t lds = lds_of(nw, ct, cv, N, Mp, np, td);
        if (lds > kLdsMax) continue;
        const double e = (double)(16 * ct / N) * N / (16 * ct) * (td ? 1.0 : 0.85);
        if (e > best + 1e-9) {
          best = e;
          p.nw = nw;
          p.ct = ct;
          p.cv = cv;
          p.tdbl = td;
          p.lds = lds;
        }
      }
    }
    p.rw = 16 * nw / N;
  };
  // complex Lnak with two k chunks needs more registers than two wavefronts per SIMD have
  if (np == 2 && Mp > 64) shape(4);
  else shape(8);
  if (((long)(W + p.rw - 1) / p.rw) * ((K + p.cv - 1) / p.cv) < cus) shape(4);
  *eff = best * p.rw * N / (16 * p.nw);
  return p;
}

Plan plan_of(int W, int M, int N, int K, int np) {
  const long cus = device_cus();
  double eff;
  Plan p = tiles_of(W, M, N, K, np, &eff);
  const long passes = (K + p.cv - 1) / p.cv, groups = (W + p.rw - 1) / p.rw;
  long best = -1;
  for (long nch = 1; nch <= passes; ++nch) {
    const long per = (passes + nch - 1) / nch;
    const long cost = ((groups * ((passes + per - 1) / per) + cus - 1) / cus) * (per + 2);
    if (best < 0 || cost < best) {
      best = cost;
      p.chunk = (int)per * p.cv;
    }
  }
  p.nchunk = (K + p.chunk - 1) / p.chunk;
  return p;
}

// Whether the kernels of k_exchange_i8w.hip take the call. Up to 16 electrons: estimated times, a constant
// and a term per walker and vector (ns, times the share of tiles that holds data for the packed product);
// more than 64 orbitals besides: not for many real products (M 128, N 16, K 640, W 1024: 734 us packed and
// 847) nor for middling numbers of complex ones (K 64, W 64: 36 and 42 us; K 384, W 64: 97 and 86). Fitted to
// 670 calls of M 16 to 128, N 3 to 16, K 8 to 640, W 1 to 1024: the choice is 0.8 % slower than the faster
// kernel in the mean, over 6 % in 1 of 20. 17 to 32 electrons: 2 x 2 tiles of complex products on more
// than 64 orbitals, unless packing saves a third of the tiles (N 28: both 23 % padding, 1570 -> 1160 us at
// M 110, K 330, W 512; N 19: 70 % of the tiles, 1010 and 1340 us at M 77, K 385) or the call is small
// (M 128, N 32, K 192, W 16: 64 and 68 us). Real trials gain little from those (mean 1 %).
bool per_walker(int W, int M, int N, int K, bool real) {
  double eff;
  tiles_of(W, M, N, K, real ? 1 : 2, &eff);
  const double pairs = (double)W * K, share = (N > 16 ? N / 32.0 : N / 16.0) * (N > 16 ? N / 32.0 : N / 16.0);
  if (N > 16) return !real && M > 64 && pairs >= 4096 && 1.5 * share > eff;
  if (M > 64 && (real ? pairs > 1e5 : pairs > 2000 && pairs < 12000)) return false;
  if (M > 64 && W < 8 && K > 500) return false;   // M 128, N 16, K 640, one walker: 34 and 41 us
  const double packed[2][2] = {{1.6, 2.8}, {1.3, 2.0}}, alone[2][2] = {{1.0, 2.0}, {1.0, 2.0}};   // ns
  const int lc = real ? 0 : 1, kc = M > 64 ? 1 : 0;
  const double base = kc ? 16.0 : (lc ? 14.0 : 12.0);
  return base + 1e-3 * alone[lc][kc] * pairs < 18.0 + 1e-3 * packed[lc][kc] * pairs * share / eff;
}

}  // namespace

bool exchange_i8_supported(int M, int N) { return N <= 32 && M <= 64 * kMaxKC; }

int exchange_i8_row(int M) { return (M + 15) / 16 * 16; }

size_t exchange_i8_bytes(int M, int N, int K, bool real) {
  return (size_t)kS * (real ? 1 : 2) * K * N * exchange_i8_row(M);
}

void exchange_i8_orders(hipStream_t s, int M, int N, int K, const double* Lnak, int* ord) {
  double* vmax = nullptr;
  AFQ_HIP(hipMalloc(&vmax, sizeof(double) * std::max(K, 1)));
  std::vector<double> h(K);
  try {
    hipLaunchKernelGGL(k_vector_max, dim3(K), dim3(256), 0, s, (long)N * M, Lnak, vmax);
    AFQ_HIP(hipGetLastError());
    AFQ_HIP(hipMemcpyAsync(h.data(), vmax, sizeof(double) * K, hipMemcpyDeviceToHost, s));
    AFQ_HIP(hipStreamSynchronize(s));
  } catch (...) {
    (void)hipFree(vmax);
    throw;
  }
  AFQ_HIP(hipFree(vmax));
  double top = 0.0;
  for (double v : h) top = std::max(top, v);
  std::vector<int> o(K, kS - 1);
  for (int n = 0; n < K; ++n) {
    if (!(top > 0.0) || !(h[n] <= top)) continue;   // zero or non-finite: keep every product
    const double r = h[n] / top;
    int on = r > 0.0 ? (int)std::ceil(5.0 + 2.0 * std::log(r) / std::log(kBase)) : 2;
    o[n] = std::min(kS - 1, std::max(N <= 16 ? 4 : 2, on));
  }
  AFQ_HIP(hipMemcpyAsync(ord, o.data(), sizeof(int) * K, hipMemcpyHostToDevice, s));
  AFQ_HIP(hipStreamSynchronize(s));
}

int exchange_i8_chunks(int W, int M, int N, int K, bool real) {
  if (per_walker(W, M, N, K, real)) return exchange_i8w_chunks(W, N, K);
  return plan_of(W, M, N, K, real ? 1 : 2).nchunk;
}

void split_lnak_i8(hipStream_t s, int M, int N, int K, const double* Lnak, bool real, int8_t* Lq,
                   double* Lu) {
  const int rows = K * N;
  hipLaunchKernelGGL(k_split_lnak_i8, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, rows, M,
                     exchange_i8_row(M), real ? 1 : 2, Lnak, Lq, Lu);
  AFQ_HIP(hipGetLastError());
}

void exchange_i8_check(int M, int N, int K) {
  AFQ_CHECK(exchange_i8_supported(M, N), AFQ_EUNSUPPORTED,
            "int8 exchange: needs N <= 32 and M <= 128");
  AFQ_CHECK((size_t)(N > 16 ? 12 : 10) * K * N * exchange_i8_row(M) < (1UL << 31), AFQ_EUNSUPPORTED,
            "int8 exchange: the Cholesky slices exceed 2 GiB");
}

void launch_exchange_i8(hipStream_t s, int W, int M, int N, int K, const double* G, bool real,
                        const int8_t* Lq, const double* Lu, const int* ord, double* Kl,
                        double* exx_part) {
  if (W <= 0 || K <= 0) return;
  exchange_i8_check(M, N, K);
  const int Mp = exchange_i8_row(M);
  AFQ_CHECK(ord != nullptr, AFQ_EINVAL, "int8 exchange: no slice orders");
  if (per_walker(W, M, N, K, real)) {
    launch_exchange_i8w(s, W, M, N, K, G, real, Lq, Lu, ord, Kl, exx_part);
    return;
  }
  const Plan p = plan_of(W, M, N, K, real ? 1 : 2);
  const dim3 grid((W + p.rw - 1) / p.rw, p.nchunk);
  auto go = [&](auto kern) {
    ensure_dynamic_lds((const void*)kern, p.lds);
    hipLaunchKernelGGL(kern, grid, dim3(64 * p.nw), p.lds, s, W, M, N, K, Mp, p.rw, p.cv, p.chunk,
                       p.tdbl, G, Lq, Lu, ord, Kl, exx_part, p.nchunk);
  };
  auto pick = [&](auto kc, auto lc) {
    constexpr int KC = decltype(kc)::value;
    constexpr bool LC = decltype(lc)::value;
    if (p.ct == 2) p.nw == 8 ? go(k_exchange_i8<KC, 2, LC, 8>) : go(k_exchange_i8<KC, 2, LC, 4>);
    else p.nw == 8 ? go(k_exchange_i8<KC, 3, LC, 8>) : go(k_exchange_i8<KC, 3, LC, 4>);
  };
  const std::integral_constant<int, 1> one;
  const std::integral_constant<int, 2> two;
  if (real) M <= 64 ? pick(one, std::false_type()) : pick(two, std::false_type());
  else if (M <= 64) pick(one, std::true_type());
  else p.ct == 2 ? go(k_exchange_i8<2, 2, true, 4>) : go(k_exchange_i8<2, 3, true, 4>);
  AFQ_HIP(hipGetLastError());
}

}  // namespace afq
