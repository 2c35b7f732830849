// Batched mixed density matrix and log-overlap of closed-shell walkers, one wavefront per walker.
//
// det_ops::MixedDensityMatrix / detail::log_overlap_impl (density_matrix.hpp:113-156, 535-601):
//   T = PsiT Phi_w                  [N,N]
//   partial pivoting (LAPACK getrf: pivot = first max of |re|+|im| in the column)
//   ov += sum_i log(+-U_ii + DBL_MIN), the sign flipped where rows were swapped, imaginary part
//        wrapped to [-pi,pi]        (log_determinant_from_getrf, determinants_impl.hpp:32-75)
//   T^-1, all zero when a pivot is exactly 0 (getri_or_zero, nda_functions.hpp:422-438)
//   G = T^-T Phi_w^T                [N,M] compact Green's function
// Optional epilogue: E1 = E0 + scl * sum_{a,j} G[a][j] haj[a][j] (Real3IndexFactorization.hpp:505-508).
//
// Both products run on FP64 MFMA 16x16x4 tiles. The inverse comes from Gauss-Jordan elimination with
// partial pivoting: its pivots are getrf's (the rows at and below step j see the same eliminations),
// so the determinant convention is unchanged. Three kernels: k_green16 (up to 16 electrons, operands
// in LDS), k_green32 (17 to 32) and k_green (up to 16 whose operands exceed 96 KB of LDS: one
// wavefront per walker; lane c holds column c of [T | I] in registers, each step broadcasts the
// pivot column through LDS).
#include "afq_internal.hpp"

#include <cfloat>

namespace afq {

namespace {

__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ inline double readlane_d(double v, int lane) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, lane);
  const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), lane);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

template <int N_>
__device__ inline double ror_d(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_update_dpp((unsigned)u, (unsigned)u, 0x120 + N_, 0xf, 0xf,
                                                  false);
  const unsigned hi = __builtin_amdgcn_update_dpp((unsigned)(u >> 32), (unsigned)(u >> 32),
                                                  0x120 + N_, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

template <int N_>
__device__ inline int ror_i(int v) {
  return __builtin_amdgcn_update_dpp(v, v, 0x120 + N_, 0xf, 0xf, false);
}

// maximum over the 16 lanes of each DPP row (every lane ends with its row's maximum; NaN is
// ignored unless a whole row is NaN)
__device__ inline double row_max16(double v) {
  v = fmax(v, ror_d<1>(v));
  v = fmax(v, ror_d<2>(v));
  v = fmax(v, ror_d<4>(v));
  v = fmax(v, ror_d<8>(v));
  return v;
}

__device__ inline int row_min16(int v) {
  v = min(v, ror_i<1>(v));
  v = min(v, ror_i<2>(v));
  v = min(v, ror_i<4>(v));
  v = min(v, ror_i<8>(v));
  return v;
}

__device__ inline int lowest_lane(unsigned long long mask) {
  return __builtin_ctzll(mask);
}

template <int NMAX>
__global__ __launch_bounds__(64) void k_green(int M, int N, const cd* __restrict__ PsiT,
                                              const cd* __restrict__ Phi, long ldw,
                                              cd* __restrict__ G, cd* __restrict__ ov,
                                              int ov_mode, double ov_scale, cd ov_add,
                                              const cd* __restrict__ haj, double E0,
                                              double e1_scale, cd* __restrict__ E, long ldE) {
  constexpr int NT = (NMAX + 15) / 16;     // 16x16 tiles along N
  constexpr int NB = 16 * NT;
  __shared__ cd sT[NB * NB];               // T, then T^-1, row-major
  __shared__ cd sCol[2][NMAX];             // pivot column broadcast (double-buffered)
  const int lane = threadIdx.x;
  const int g = lane >> 4, r16 = lane & 15;
  const int w = blockIdx.x;
  const cd* P = Phi + (long)w * ldw;
  const bool want_e1 = E != nullptr && haj != nullptr;

  // ---- T[a][c] = sum_i PsiT[a][i] Phi[i][c]  (MFMA; k = orbital i) ----
  {
    d4 tr[NT][NT], ti[NT][NT];
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int b = 0; b < NT; ++b) {
        tr[a][b] = d4{0, 0, 0, 0};
        ti[a][b] = d4{0, 0, 0, 0};
      }
    for (int k0 = 0; k0 < M; k0 += 16) {
      double ar[NT][4], ai[NT][4], br[NT][4], bi[NT][4];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int a = t * 16 + r16;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int k = k0 + 4 * g + s;
          const cd x = (a < N && k < M) ? PsiT[(long)a * M + k] : cmk(0, 0);
          ar[t][s] = x.re;
          ai[t][s] = x.im;
          const int c = t * 16 + r16;
          const cd y = (c < N && k < M) ? P[(long)k * N + c] : cmk(0, 0);
          br[t][s] = y.re;
          bi[t][s] = y.im;
        }
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
#pragma unroll
        for (int a = 0; a < NT; ++a)
#pragma unroll
          for (int b = 0; b < NT; ++b) {
            tr[a][b] = mfma16x16x4(ar[a][s], br[b][s], tr[a][b]);
            ti[a][b] = mfma16x16x4(ar[a][s], bi[b][s], ti[a][b]);
          }
#pragma unroll
        for (int a = 0; a < NT; ++a)
#pragma unroll
          for (int b = 0; b < NT; ++b) {
            tr[a][b] = mfma16x16x4(-ai[a][s], bi[b][s], tr[a][b]);
            ti[a][b] = mfma16x16x4(ai[a][s], br[b][s], ti[a][b]);
          }
      }
    }
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          sT[(a * 16 + acc_row<double>(g, r)) * NB + b * 16 + r16] = cmk(tr[a][b][r], ti[a][b][r]);
  }
  wave_sync();

  // ---- Gauss-Jordan on [T | I]: lane c < 2N holds column c ----
  cd x[NMAX];
#pragma unroll
  for (int r = 0; r < NMAX; ++r) {
    cd v = cmk(0.0, 0.0);
    if (r < N) {
      if (lane < N) v = sT[r * NB + lane];
      else if (lane - N == r) v = cmk(1.0, 0.0);
    }
    x[r] = v;
  }
  cd upiv = cmk(1.0, 0.0);     // lane j keeps +-U_jj; the logs are taken in parallel afterwards
  bool singular = false;
  {
    // Step j is unrolled, so column j is a register of lane j: lane j finds the pivot in its own
    // column (izamax: first maximum of |re|+|im| from row j down) and readlane broadcasts it; the
    // row swap selects over a static row range; lane j publishes its swapped column to LDS, from
    // which every lane reads the multipliers at fixed addresses (one LDS round trip per step,
    // double-buffered so that the next step's write cannot race this step's reads).
#pragma unroll
    for (int j = 0; j < NMAX; ++j) {
      bool go = j < N;
      double best = cabs1(x[j]);
      int bi = j;
#pragma unroll
      for (int r = j + 1; r < NMAX; ++r) {
        if (r < N) {
          const double v = cabs1(x[r]);
          if (v > best) {
            best = v;
            bi = r;
          }
        }
      }
      const int p = __builtin_amdgcn_readlane(bi, j);
      cd xp = x[j];
#pragma unroll
      for (int r = j + 1; r < NMAX; ++r)
        if (r == p) xp = x[r];
      const cd piv = cmk(readlane_d(xp.re, j), readlane_d(xp.im, j));
      if (go && lane == j) upiv = (p == j) ? piv : -piv;   // the sign flips where the pivot row moved
      if (go && cis0(piv)) {
        singular = true;   // getrf records the zero pivot and goes on; getri_or_zero zeroes T^-1
        go = false;
      }
      if (go) {
        if (p != j) {
#pragma unroll
          for (int r = j + 1; r < NMAX; ++r)
            if (r == p) x[r] = x[j];
          x[j] = xp;
        }
        cd* col = sCol[j & 1];
        if (lane == j)
#pragma unroll
          for (int r = 0; r < NMAX; ++r)
            if (r < N) col[r] = x[r];
        wave_sync();
        const cd xjn = x[j] * cdiv(cmk(1.0, 0.0), piv);
#pragma unroll
        for (int r = 0; r < NMAX; ++r) {
          if (r < N && r != j) {
            const cd f = col[r];
            if (!cis0(f)) x[r] -= f * xjn;
          }
        }
        x[j] = xjn;
      }
    }
  }

  // sum_j log(+-U_jj + DBL_MIN): one log per lane, then a wavefront sum
  cd acc = (lane < N) ? clog_(cmk(upiv.re + DBL_MIN, upiv.im)) : cmk(0.0, 0.0);
  for (int off = 32; off > 0; off >>= 1) {
    acc.re += __shfl_xor(acc.re, off, 64);
    acc.im += __shfl_xor(acc.im, off, 64);
  }
  if (lane == 0) {
    if (ov_mode == 2) acc += ov[w];
    const double pi = 3.14159265358979323846;
    // the reference loops until the value is in range; a non-finite value would never get
    // there, so only finite values are wrapped
    if (!isfinite(acc.im)) {
    } else if (acc.im > pi) {
      while (acc.im > pi) acc.im -= 2 * pi;
    } else if (acc.im < -pi) {
      while (acc.im < -pi) acc.im += 2 * pi;
    }
    if (ov_mode != 0) ov[w] = ov_scale * acc + ov_add;
  }
  if (G == nullptr && E == nullptr) return;

  // ---- T^-1 to LDS as [b][a] (zero padded to NB x NB) ----
  wave_sync();
  for (int e = lane; e < NB * NB; e += 64) sT[e] = cmk(0, 0);
  wave_sync();
  if (lane >= N && lane < 2 * N && !singular) {
    const int a = lane - N;
#pragma unroll
    for (int r = 0; r < NMAX; ++r)
      if (r < N) sT[r * NB + a] = x[r];
  }
  wave_sync();

  // ---- G[a][i] = sum_b Tinv[b][a] Phi[i][b]  (MFMA; rows a, cols i, k = b) ----
  cd e1 = cmk(0.0, 0.0);
  cd* Gw = G ? G + (long)w * N * M : nullptr;
  for (int i0 = 0; i0 < M; i0 += 16) {
    d4 gr[NT], gi[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      gr[t] = d4{0, 0, 0, 0};
      gi[t] = d4{0, 0, 0, 0};
    }
    const int i = i0 + r16;
#pragma unroll
    for (int b0 = 0; b0 < NB; b0 += 16) {
      double ar[NT][4], ai[NT][4], br[4], bi[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int b = b0 + 4 * g + s;
        const cd y = (i < M && b < N) ? P[(long)i * N + b] : cmk(0, 0);
        br[s] = y.re;
        bi[s] = y.im;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const cd z = sT[b * NB + t * 16 + r16];   // Tinv^T[a][b] = Tinv[b][a]
          ar[t][s] = z.re;
          ai[t][s] = z.im;
        }
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          gr[t] = mfma16x16x4(ar[t][s], br[s], gr[t]);
          gi[t] = mfma16x16x4(ar[t][s], bi[s], gi[t]);
          gr[t] = mfma16x16x4(-ai[t][s], bi[s], gr[t]);
          gi[t] = mfma16x16x4(ai[t][s], br[s], gi[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int a = t * 16 + acc_row<double>(g, r);
        if (a < N && i < M) {
          const cd v = cmk(gr[t][r], gi[t][r]);
          if (Gw) Gw[(long)a * M + i] = v;
          if (want_e1) e1 += v * haj[(long)a * M + i];
        }
      }
  }
  if (want_e1) {
    for (int off = 32; off > 0; off >>= 1) {
      e1.re += __shfl_xor(e1.re, off, 64);
      e1.im += __shfl_xor(e1.im, off, 64);
    }
    if (lane == 0) E[(long)w * ldE] = cmk(E0, 0.0) + e1_scale * e1;
  }
}


// ---- N <= 16 with the operands staged in LDS: four wavefronts per walker ----
//
// The one-wavefront kernel above runs a serial chain per walker, and a batch of a few hundred
// walkers leaves most SIMDs idle, so its time is that chain's latency. Here a 256-thread
// workgroup shares the walker's work:
//   * all 256 threads stage Phi_w [M][N+1], PsiT [N][M+1] and haj [N][M] in one batch of loads
//     (rows padded so that the 16 rows an MFMA fragment reads fall into distinct banks);
//   * T = PsiT Phi_w is split over k: wavefront v takes the 16-wide k chunks v, v+4, ..., and
//     wavefront 0 sums the four partial tiles in a fixed order;
//   * wavefront 0 inverts T by Gauss-Jordan in a row layout that keeps all 64 lanes busy: lane
//     (r, h) = (lane % 16, lane / 16) holds columns 8h..8h+7 of row r of [T | I] (T in columns
//     0..15, I in 16..31). Rows are never moved: each row carries its getrf position, the pivot
//     is chosen with izamax's rule over the rows at positions >= j (first maximum of |re|+|im|
//     by position; a NaN at position j is kept, a later NaN is skipped), and positions are
//     swapped as getrf swaps rows. The row at position j is then the pivot row of step j, so
//     the eliminations, pivots and signs are getrf's. Each step is one 16-lane DPP maximum,
//     a few readlanes and one LDS round trip for the pivot row and the multipliers;
//   * wavefronts 1-3 compute the 16 x 16 tiles of G (and the E1 partial sums) while wavefront 0
//     takes the logarithms of the pivots.
constexpr int kGWaves = 4;

// e = q d + rem for 0 <= e < 2^24 and 0 < d, from a float estimate corrected by one step
__device__ inline void divmod(int e, int d, float rcp, int& q, int& rem) {
  q = (int)((float)e * rcp);
  rem = e - q * d;
  if (rem < 0) {
    --q;
    rem += d;
  } else if (rem >= d) {
    ++q;
    rem -= d;
  }
}

__global__ __launch_bounds__(64 * kGWaves) void k_green16(
    int M, int N, const cd* __restrict__ PsiT, const cd* __restrict__ Phi, long ldw,
    cd* __restrict__ G, cd* __restrict__ ov, int ov_mode, double ov_scale, cd ov_add,
    const cd* __restrict__ haj, double E0, double e1_scale, cd* __restrict__ E, long ldE) {
  __shared__ cd sPart[kGWaves * 256];      // partial T tiles [wave][a][c]; later T^-1 [b][a]
  __shared__ cd sRow[2][32];               // pivot row of the step (double-buffered)
  __shared__ cd sF[2][16];                 // column j of every row (double-buffered)
  __shared__ cd sE[kGWaves];
  extern __shared__ cd sDyn[];             // Phi_w [M][N+1], PsiT [N][M+1], haj [N][M]
  const int tid = threadIdx.x;
  const int lane = tid & 63, wv = tid >> 6;
  const int g = lane >> 4, r16 = lane & 15;
  const int w = blockIdx.x;
  const bool want_e1 = E != nullptr && haj != nullptr;
  const int ldp = N + 1, ldq = M + 1;
  cd* sPhi = sDyn;
  cd* sPs = sDyn + M * ldp;
  cd* sH = sPs + N * ldq;

  // ---- staging: every load of a batch in flight before the first LDS write ----
  {
    const cd* Pg = Phi + (long)w * ldw;
    const int mn = M * N;
    const int tot = (want_e1 ? 3 : 2) * mn;
    constexpr int B = 12;
    const float rn = 1.0f / (float)N, rm = 1.0f / (float)M;
    for (int e0 = 0; e0 < tot; e0 += 256 * B) {
      double2 v[B];
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const int e = min(e0 + 256 * b + tid, tot - 1);
        const cd* src = e < mn ? Pg + e : (e < 2 * mn ? PsiT + (e - mn) : haj + (e - 2 * mn));
        v[b] = *reinterpret_cast<const double2*>(src);
      }
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const int e = e0 + 256 * b + tid;
        if (e < tot) {
          cd* dst;
          int row, col;
          if (e < mn) {
            divmod(e, N, rn, row, col);
            dst = sPhi + row * ldp + col;
          } else if (e < 2 * mn) {
            divmod(e - mn, M, rm, row, col);
            dst = sPs + row * ldq + col;
          } else {
            dst = sH + (e - 2 * mn);
          }
          *reinterpret_cast<double2*>(dst) = v[b];
        }
      }
    }
  }
  __syncthreads();

  // ---- partial T[a][c] = sum_{i in this wavefront's chunks} PsiT[a][i] Phi[i][c] ----
  {
    d4 tra = d4{0, 0, 0, 0}, trb = d4{0, 0, 0, 0}, tia = d4{0, 0, 0, 0}, tib = d4{0, 0, 0, 0};
    for (int k0 = 16 * wv; k0 < M; k0 += 16 * kGWaves) {
      double ar[4], ai[4], br[4], bi[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int k = k0 + 4 * g + s;
        const cd x = (r16 < N && k < M) ? sPs[r16 * ldq + k] : cmk(0, 0);
        const cd y = (r16 < N && k < M) ? sPhi[k * ldp + r16] : cmk(0, 0);
        ar[s] = x.re;
        ai[s] = x.im;
        br[s] = y.re;
        bi[s] = y.im;
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        tra = mfma16x16x4(ar[s], br[s], tra);
        trb = mfma16x16x4(-ai[s], bi[s], trb);
        tia = mfma16x16x4(ar[s], bi[s], tia);
        tib = mfma16x16x4(ai[s], br[s], tib);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
      sPart[wv * 256 + acc_row<double>(g, r) * 16 + r16] =
          cmk(tra[r] + trb[r], tia[r] + tib[r]);
  }
  __syncthreads();

  cd upiv = cmk(1.0, 0.0);     // lane j < N: +-U_jj
  if (wv == 0) {
    const int r = r16, h = g;
    cd x[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int c = 8 * h + q;
      cd v = cmk(0.0, 0.0);
      if (h < 2) {
        if (r < N && c < N) {
          const int e = r * 16 + c;
          v = ((sPart[e] + sPart[256 + e]) + sPart[512 + e]) + sPart[768 + e];
        }
      } else if (r < N && c - 16 == r) {
        v = cmk(1.0, 0.0);
      }
      x[q] = v;
    }
    int pos = r;                 // getrf position of row r
    bool singular = false;
    // steps j >= N do nothing: a uniform branch rather than a break, so that the loop unrolls
    // and x[] stays in registers
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      if (j < N) {
        const int hj = j >> 3, qj = j & 7;
        const bool cand = h == hj && r < N && pos >= j;
        const double v = cand ? cabs1(x[qj]) : -1.0;
        // the row now at position j, and izamax's choice
        const int q = lowest_lane(__ballot(h == 0 && pos == j));
        const double vq = readlane_d(v, q + 16 * hj);
        int p;
        if (isnan(vq)) {
          p = q;
        } else {
          const double m = row_max16(v);
          const unsigned long long mask = __ballot(cand && v == m);
          if (__builtin_popcountll(mask) == 1) {
            p = lowest_lane(mask) - 16 * hj;
          } else {
            const int kmin = row_min16(((mask >> lane) & 1ull) ? pos : 0x7fffffff);
            const int km = __builtin_amdgcn_readlane(kmin, 16 * hj);
            p = lowest_lane(__ballot(h == 0 && pos == km));
          }
        }
        p = __builtin_amdgcn_readfirstlane(p);
        const int lp = p + 16 * hj;
        const cd piv = cmk(readlane_d(x[qj].re, lp), readlane_d(x[qj].im, lp));
        const int pp = __builtin_amdgcn_readlane(pos, lp);
        if (lane == j) upiv = (pp == j) ? piv : -piv;   // the sign flips where getrf swaps rows
        if (cis0(piv)) {
          singular = true;   // getrf records the zero pivot and goes on; getri_or_zero zeroes it
        } else {
          if (r == q) pos = pp;
          if (r == p) pos = j;
          cd* row = sRow[j & 1];
          cd* fv = sF[j & 1];
          if (r == p)
#pragma unroll
            for (int e = 0; e < 8; ++e) row[8 * h + e] = x[e];
          if (h == hj) fv[r] = x[qj];
          wave_sync();
          const cd inv = cdiv(cmk(1.0, 0.0), piv);
          cd pr[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) pr[e] = row[8 * h + e];
          const cd f = fv[r];
          if (r == p) {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = pr[e] * inv;
          } else if (!cis0(f)) {
            const cd mlt = f * inv;
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] -= mlt * pr[e];
          }
        }
      }
    }
    // row r is row pos of [I | T^-1]: T^-1 to LDS as [b][a]
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (h >= 2) {
        const int c = 8 * (h - 2) + e;
        sPart[pos * 16 + c] = (!singular && r < N && c < N) ? x[e] : cmk(0.0, 0.0);
      }
    }
  }
  __syncthreads();

  if (wv == 0) {
    // sum_j log(+-U_jj + DBL_MIN): one log per lane, then a wavefront sum
    cd acc = (lane < N) ? clog_(cmk(upiv.re + DBL_MIN, upiv.im)) : cmk(0.0, 0.0);
    for (int off = 32; off > 0; off >>= 1) {
      acc.re += __shfl_xor(acc.re, off, 64);
      acc.im += __shfl_xor(acc.im, off, 64);
    }
    if (lane == 0) {
      if (ov_mode == 2) acc += ov[w];
      const double pi = 3.14159265358979323846;
      // the reference loops until the value is in range; a non-finite value would never get
      // there, so only finite values are wrapped
      if (!isfinite(acc.im)) {
      } else if (acc.im > pi) {
        while (acc.im > pi) acc.im -= 2 * pi;
      } else if (acc.im < -pi) {
        while (acc.im < -pi) acc.im += 2 * pi;
      }
      if (ov_mode != 0) ov[w] = ov_scale * acc + ov_add;
    }
  }
  if (G == nullptr && E == nullptr) return;

  // ---- G[a][i] = sum_b Tinv[b][a] Phi[i][b], one 16-column tile of i per step ----
  cd e1 = cmk(0.0, 0.0);
  cd* Gw = G ? G + (long)w * N * M : nullptr;
  if (wv > 0) {
    for (int i0 = 16 * (wv - 1); i0 < M; i0 += 16 * (kGWaves - 1)) {
      d4 gra = d4{0, 0, 0, 0}, grb = d4{0, 0, 0, 0}, gia = d4{0, 0, 0, 0}, gib = d4{0, 0, 0, 0};
      const int i = i0 + r16;
      double tr_[4], ti_[4], pr_[4], pi_[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int b = 4 * g + s;
        const cd y = (i < M && b < N) ? sPhi[i * ldp + b] : cmk(0, 0);
        pr_[s] = y.re;
        pi_[s] = y.im;
        const cd z = sPart[b * 16 + r16];            // Tinv^T[a][b] = Tinv[b][a]
        tr_[s] = z.re;
        ti_[s] = z.im;
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        gra = mfma16x16x4(tr_[s], pr_[s], gra);
        grb = mfma16x16x4(-ti_[s], pi_[s], grb);
        gia = mfma16x16x4(tr_[s], pi_[s], gia);
        gib = mfma16x16x4(ti_[s], pr_[s], gib);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int a = acc_row<double>(g, r);
        if (a < N && i < M) {
          const cd v = cmk(gra[r] + grb[r], gia[r] + gib[r]);
          if (Gw) Gw[(long)a * M + i] = v;
          if (want_e1) e1 += v * sH[a * M + i];
        }
      }
    }
  }
  if (want_e1) {
    for (int off = 32; off > 0; off >>= 1) {
      e1.re += __shfl_xor(e1.re, off, 64);
      e1.im += __shfl_xor(e1.im, off, 64);
    }
    if (lane == 0) sE[wv] = e1;
    __syncthreads();
    if (tid == 0) E[(long)w * ldE] = cmk(E0, 0.0) + e1_scale * ((sE[1] + sE[2]) + sE[3]);
  }
}

// ---- 17 to 32 electrons: four wavefronts per walker, the inverse in place ----
//
// T = PsiT Phi_w on MFMA, its k range (orbitals) dealt to the wavefronts in steps of four, operands
// straight from memory (Phi_w is read twice, 16 lanes along a row each time, rather than held in
// LDS, so that four workgroups fit a CU); the partial tiles are added in a fixed order. The Gauss-Jordan
// elimination works in place: 8 threads hold column c (rows q, q + 8, q + 16, q + 24) and the column of
// step j becomes the inverse's column of its pivot row, which is what [T | I] gives with half of the
// columns. A step is one barrier: the owners of column j choose the pivot (izamax's rule over
// the rows at getrf positions >= j: first maximum of |re| + |im| by position; a NaN at position j is
// kept, a later NaN skipped) and publish the column, the pivot's position and its reciprocal;
// every thread takes the pivot row's entry of its column from the 8 lanes through DPP. Rows
// never move: each carries its getrf position. The loop stays rolled (the fully unrolled single-
// wavefront elimination it replaces streamed ~100 KB of code per walker). Bound by the latency of
// the serial steps. M 128, N 32, 1024 walkers: 188 -> 120 us (G and overlap), 130 -> 86 us (overlap
// alone); M 88, N 22, 137 walkers 107 -> 45 us; M 77, N 19, 201 walkers 85 -> 40 us.
// the bits of the one lane whose v is not all zeros
template <int CTRL>
__device__ inline double dpp8_or(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_update_dpp((unsigned)u, (unsigned)u, CTRL, 0xf, 0xf, false);
  const unsigned hi = __builtin_amdgcn_update_dpp((unsigned)(u >> 32), (unsigned)(u >> 32), CTRL, 0xf,
                                                  0xf, false);
  return __builtin_bit_cast(double, u | ((unsigned long long)hi << 32 | lo));
}
template <int CTRL>
__device__ inline double dpp8_max(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_update_dpp((unsigned)u, (unsigned)u, CTRL, 0xf, 0xf, false);
  const unsigned hi = __builtin_amdgcn_update_dpp((unsigned)(u >> 32), (unsigned)(u >> 32), CTRL, 0xf,
                                                  0xf, false);
  return fmax(v, __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo));
}
template <int CTRL>
__device__ inline int dpp8_min(int v) {
  return min(v, __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false));
}
// over the 8 lanes of a column: quad permutes (lanes ^1, ^2), then the other quad (half-row mirror)
__device__ inline double only8(double v) { return dpp8_or<0x141>(dpp8_or<0x4E>(dpp8_or<0xB1>(v))); }
__device__ inline double max8(double v) { return dpp8_max<0x141>(dpp8_max<0x4E>(dpp8_max<0xB1>(v))); }
__device__ inline int min8(int v) { return dpp8_min<0x141>(dpp8_min<0x4E>(dpp8_min<0xB1>(v))); }

__global__ __launch_bounds__(256, 4) void k_green32(
    int M, int N, const cd* __restrict__ PsiT, const cd* __restrict__ Phi, long ldw,
    cd* __restrict__ G, cd* __restrict__ ov, int ov_mode, double ov_scale, cd ov_add,
    const cd* __restrict__ haj, double E0, double e1_scale, cd* __restrict__ E, long ldE) {
  constexpr int NB = 32, LD = 33;
  __shared__ cd sT[2][NB * LD];            // partial T tiles; then [0]: T, later T^-1 [b][a]
  __shared__ cd sF[2][NB];                 // column j of every row
  __shared__ cd sInv[2];                   // 1 / pivot
  __shared__ int sPos[2];                  // the pivot's position; -1: the pivot is exactly zero
  __shared__ cd sPiv[NB];                  // +-U_jj
  __shared__ int sRow[NB];                 // pivot row of step j
  __shared__ cd sE[4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int w = blockIdx.x;
  const cd* P = Phi + (long)w * ldw;
  const bool inverse = G != nullptr || E != nullptr;

  // ---- partial T[a][c] over this wavefront's k steps ----
  {
    d4 tr[2][2], ti[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        tr[a][b] = d4{0, 0, 0, 0};
        ti[a][b] = d4{0, 0, 0, 0};
      }
    const int steps = (M + 3) >> 2;
    auto load = [&](int t, cd (&x)[2], cd (&y)[2]) {
      const int k = 4 * t + g;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int r = 16 * u + r16;
        const bool ok = r < N && k < M;
        x[u] = ok ? PsiT[r * M + k] : cmk(0, 0);
        y[u] = ok ? P[k * N + r] : cmk(0, 0);
      }
    };
    cd x[2], y[2];
    load(wv, x, y);
    for (int t = wv; t < steps; t += 4) {   // the next step's operands are loaded ahead
      cd nx[2], ny[2];
      load(t + 4, nx, ny);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          tr[a][b] = mfma16x16x4(x[a].re, y[b].re, tr[a][b]);
          ti[a][b] = mfma16x16x4(x[a].re, y[b].im, ti[a][b]);
        }
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          tr[a][b] = mfma16x16x4(-x[a].im, y[b].im, tr[a][b]);
          ti[a][b] = mfma16x16x4(x[a].im, y[b].re, ti[a][b]);
        }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        x[u] = nx[u];
        y[u] = ny[u];
      }
    }
    // wavefronts 2, 3 into [0], [1]; 0 and 1 add theirs; 1 into [1]; 0 adds it
    auto put = [&](cd* dst, const cd* add) {
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int e = (16 * a + acc_row<double>(g, r)) * LD + 16 * b + r16;
            cd v = cmk(tr[a][b][r], ti[a][b][r]);
            if (add) v = add[e] + v;
            dst[e] = v;
          }
    };
    if (wv >= 2) put(sT[wv - 2], nullptr);
    __syncthreads();
    if (wv < 2) put(sT[wv], sT[wv]);
    __syncthreads();
  }
  // ---- in-place Gauss-Jordan: thread (c, q) holds rows q + 8 i of column c ----
  const int c = tid >> 3, q = tid & 7;
  cd x[4];
  int pos[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = q + 8 * i;
    pos[i] = r;
    x[i] = (r < N && c < N) ? sT[0][r * LD + c] + sT[1][r * LD + c] : cmk(0.0, 0.0);
  }
  // the owners of column j choose its pivot and publish the column
  auto publish = [&](int j) {
    double m = -1.0, vq = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double v = cabs1(x[i]);
      if (q + 8 * i < N && pos[i] >= j) m = fmax(m, v);   // drops a NaN
      if (pos[i] == j) vq = v;
    }
    m = max8(m);
    vq = only8(vq);                                        // the row at position j
    int k = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (q + 8 * i < N && pos[i] >= j && cabs1(x[i]) == m) k = min(k, pos[i]);
    k = min8(k);
    if (isnan(vq)) k = j;
    cd pv = cmk(0.0, 0.0);
    int row = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (pos[i] == k) {
        pv = x[i];
        row = q + 8 * i;
      }
    row = min8(row);
    pv.re = only8(pv.re);
    pv.im = only8(pv.im);
    const bool zero = cis0(pv);
    const cd inv = zero ? cmk(0.0, 0.0) : cdiv(cmk(1.0, 0.0), pv);
#pragma unroll
    for (int i = 0; i < 4; ++i) sF[j & 1][q + 8 * i] = x[i];
    if (q == 0) {
      sInv[j & 1] = inv;
      sPos[j & 1] = zero ? -1 : k;
      sPiv[j] = k == j ? pv : -pv;   // the sign flips where getrf swaps rows
      sRow[j] = row;
    }
  };
  if (c == 0) publish(0);
  __syncthreads();
  bool singular = false;
  for (int j = 0; j < N; ++j) {
    const int k = sPos[j & 1];
    if (k < 0) {
      singular = true;   // getrf records the zero pivot and goes on; getri_or_zero zeroes T^-1
    } else if (c < N && (inverse || c > j)) {
      const cd inv = sInv[j & 1];
      cd p = cmk(0.0, 0.0), f[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f[i] = sF[j & 1][q + 8 * i];
        if (pos[i] == k) p = x[i];
      }
      p.re = only8(p.re);
      p.im = only8(p.im);
      if (c == j) p = cmk(1.0, 0.0);   // the identity's column of the pivot row takes this place
      p = p * inv;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const cd old = c == j ? cmk(0.0, 0.0) : x[i];
        x[i] = pos[i] == k ? p : (cis0(f[i]) ? old : old - f[i] * p);
      }
    }
    if (k >= 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) pos[i] = pos[i] == k ? j : (pos[i] == j ? k : pos[i]);
    }
    if (c == j + 1 && c < N) publish(j + 1);
    __syncthreads();
  }

  if (wv == 0) {
    // sum_j log(+-U_jj + DBL_MIN): one log per lane, then a wavefront sum
    cd acc = (lane < N) ? clog_(cmk(sPiv[lane].re + DBL_MIN, sPiv[lane].im)) : cmk(0.0, 0.0);
    for (int off = 32; off > 0; off >>= 1) {
      acc.re += __shfl_xor(acc.re, off, 64);
      acc.im += __shfl_xor(acc.im, off, 64);
    }
    if (lane == 0) {
      if (ov_mode == 2) acc += ov[w];
      const double pi = 3.14159265358979323846;
      // the reference loops until the value is in range; a non-finite value would never get
      // there, so only finite values are wrapped
      if (!isfinite(acc.im)) {
      } else if (acc.im > pi) {
        while (acc.im > pi) acc.im -= 2 * pi;
      } else if (acc.im < -pi) {
        while (acc.im < -pi) acc.im += 2 * pi;
      }
      if (ov_mode != 0) ov[w] = ov_scale * acc + ov_add;
    }
  }
  if (!inverse) return;

  // ---- T^-1 to LDS as [b][a]: row r ends at position pos, column slot j is pivot row sRow[j]'s ----
  cd* sI = sT[0];
  if (c < N)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (q + 8 * i < N) sI[pos[i] * LD + sRow[c]] = singular ? cmk(0.0, 0.0) : x[i];
  for (int e = tid; e < NB * NB; e += 256) {
    const int b = e / NB, a = e % NB;
    if (b >= N || a >= N) sI[b * LD + a] = cmk(0.0, 0.0);
  }
  __syncthreads();

  // ---- G[a][i] = sum_b Tinv[b][a] Phi[i][b], 16 columns i per wavefront and turn ----
  const bool want_e1 = E != nullptr && haj != nullptr;
  cd e1 = cmk(0.0, 0.0);
  cd* Gw = G ? G + (long)w * N * M : nullptr;
  for (int i0 = 16 * wv; i0 < M; i0 += 64) {
    asm volatile("" ::: "memory");   // T^-1 is read from LDS in every turn: hoisted, it would spill
    const int i = i0 + r16;
    d4 gr[2], gi[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      gr[t] = d4{0, 0, 0, 0};
      gi[t] = d4{0, 0, 0, 0};
    }
    cd y[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int b = 4 * s + g;
      y[s] = (i < M && b < N) ? P[(long)i * N + b] : cmk(0, 0);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      cd z[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) z[t] = sI[(4 * s + g) * LD + 16 * t + r16];   // Tinv^T[a][b]
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        gr[t] = mfma16x16x4(z[t].re, y[s].re, gr[t]);
        gi[t] = mfma16x16x4(z[t].re, y[s].im, gi[t]);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        gr[t] = mfma16x16x4(-z[t].im, y[s].im, gr[t]);
        gi[t] = mfma16x16x4(z[t].im, y[s].re, gi[t]);
      }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int a = 16 * t + acc_row<double>(g, r);
        if (a < N && i < M) {
          const cd v = cmk(gr[t][r], gi[t][r]);
          if (Gw) Gw[(long)a * M + i] = v;
          if (want_e1) e1 += v * haj[(long)a * M + i];
        }
      }
  }
  if (want_e1) {
    for (int off = 32; off > 0; off >>= 1) {
      e1.re += __shfl_xor(e1.re, off, 64);
      e1.im += __shfl_xor(e1.im, off, 64);
    }
    if (lane == 0) sE[wv] = e1;
    __syncthreads();
    if (tid == 0) E[(long)w * ldE] = cmk(E0, 0.0) + e1_scale * ((sE[0] + sE[1]) + (sE[2] + sE[3]));
  }
}

}  // namespace

void launch_green(hipStream_t s, int nb, int M, int N, const double* PsiT, const double* Phi,
                  long ldw, double* G, double* ov, int ov_mode, double ov_scale, cd ov_add,
                  const double* haj, double E0, double e1_scale, double* E, long ldE) {
  if (nb <= 0 || N <= 0) return;
  AFQ_CHECK(N <= 32, AFQ_EUNSUPPORTED, "mixed density matrix: more than 32 electrons per spin");
  const bool e1 = E != nullptr && haj != nullptr;
  // N <= 16: four wavefronts per walker when Phi_w, PsiT and haj (rows padded) fit in 96 KB
  const size_t lds16 = sizeof(cd) * ((size_t)M * (N + 1) + (size_t)N * (M + 1) +
                                     (e1 ? (size_t)M * N : 0));
  if (N <= 16 && lds16 <= 96 * 1024) {
    ensure_dynamic_lds((const void*)k_green16, lds16);
    hipLaunchKernelGGL(k_green16, dim3(nb), dim3(64 * kGWaves), lds16, s, M, N,
                       reinterpret_cast<const cd*>(PsiT), reinterpret_cast<const cd*>(Phi), ldw,
                       reinterpret_cast<cd*>(G), reinterpret_cast<cd*>(ov), ov_mode, ov_scale,
                       ov_add, reinterpret_cast<const cd*>(haj), E0, e1_scale,
                       reinterpret_cast<cd*>(E), ldE);
    AFQ_HIP(hipGetLastError());
    return;
  }
  if (N > 16) {
    hipLaunchKernelGGL(k_green32, dim3(nb), dim3(256), 0, s, M, N, reinterpret_cast<const cd*>(PsiT),
                       reinterpret_cast<const cd*>(Phi), ldw, reinterpret_cast<cd*>(G),
                       reinterpret_cast<cd*>(ov), ov_mode, ov_scale, ov_add,
                       reinterpret_cast<const cd*>(haj), E0, e1_scale, reinterpret_cast<cd*>(E), ldE);
    AFQ_HIP(hipGetLastError());
    return;
  }
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(nb), dim3(64), 0, s, M, N, reinterpret_cast<const cd*>(PsiT),
                       reinterpret_cast<const cd*>(Phi), ldw, reinterpret_cast<cd*>(G),
                       reinterpret_cast<cd*>(ov), ov_mode, ov_scale, ov_add,
                       reinterpret_cast<const cd*>(haj), E0, e1_scale, reinterpret_cast<cd*>(E), ldE);
  };
  if (N <= 8) go(k_green<8>);
  else go(k_green<16>);
  AFQ_HIP(hipGetLastError());
}

}  // namespace afq
