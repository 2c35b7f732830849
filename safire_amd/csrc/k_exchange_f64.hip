// Exchange and Coulomb contraction of the plain FP64 form for up to 128 orbitals
// (Real3IndexFactorization::energy_impl, Real3IndexFactorization.hpp:476-559):
//
//   T_wn[b][a] = sum_k G_w[b][k] Lnak[n][a][k],  sum_ab T_ab T_ba per walker,  Kl_wn = sum_a T_aa
//
// as one product of the flat row sets (w, b) and (n, a), both contiguous in memory, so that 16-wide
// MFMA tiles are filled across walkers and across Cholesky vectors: a workgroup takes Rw walkers
// (Rw N <= 16 NW rows) and, per pass, Cv vectors (Cv N <= 16 CT columns). A walker of 19 electrons
// then uses 89 % of the rows and columns of its tiles; padded to 2 x 2 tiles it would use 35 %.
//
// Each wavefront keeps its 16 rows of G in registers for its whole life (up to 128 VGPR pairs at
// M = 128), so G is read once; the columns are staged through LDS in k slices of 128 bytes a row, double
// buffered, one barrier per slice, and shared by the NW wavefronts. The T block of a pass goes to
// LDS once, where all threads form the products T_ab T_ba. The two wavefronts of a SIMD take that
// epilogue at different slices of the next pass (the second half of the wavefronts half a pass
// later), so that one's LDS and VALU work runs under the other's MFMAs.
//
// Real trial orbitals give Lnak an exactly zero imaginary part. Lnak then comes as a real array
// (LC = false, rows zero-padded to ldl) and a complex tile takes 2 FP64 MFMAs per k step, not 4. A
// row of G with a NaN or Inf makes its whole T row NaN in either form (with complex products the
// zeros of Im L do that; here the element is made NaN when it is loaded).
//
// Bound: FP64 MFMA (64 cycles per 16x16x4 on a SIMD). Per launch, against the kernel of k_energy.hip
// that pads every N x N block and re-reads G per pair of vectors (it stays for M > 128):
//   M 128, N 32, K 640, 1024 walkers, real trial     19.2 -> 6.5 ms (73 % of what an 8192^3 FP64 GEMM reaches)
//   M 77, N 19, K 385, 201 walkers, complex trial     1.27 -> 0.49 ms
//   M 24, N 6, K 96, 64 walkers, real trial           27.9 -> 8.0 us
// The first two now take the quadratic form over the pair table instead (k_gemm_real.hip); this kernel
// runs the small calls and those with few vectors per orbital, where it is the faster one.
#include "afq_internal.hpp"

#include <algorithm>

namespace afq {

namespace {

template <int KCH, int CT, bool LC, int NW>
__global__ __launch_bounds__(64 * NW, NW / 4) void k_exchange_f64(
    int W, int M, int N, int K, int ldl, int Rw, int Cv, int chunk, const double* __restrict__ G,
    const double* __restrict__ L, double* __restrict__ Kl, double* __restrict__ part, int nchunk) {
  constexpr int kThreads = 64 * NW;
  constexpr int kCols = 16 * CT;
  constexpr int EB = LC ? 16 : 8;                 // bytes of an element of L
  constexpr int kKS = LC ? 8 : 16;                // k slice: 128 bytes of a row
  constexpr int SPS = kKS / 4;                    // MFMA k steps of a slice
  constexpr int NS = KCH * 16 / kKS;              // slices of the longest row
  constexpr int ROWB = kKS * EB + 16;             // staged row: odd multiple of 16 bytes
  constexpr int TPR = kKS * EB / 16;              // 16-byte pieces per staged row
  constexpr int PCS = (kCols * TPR + kThreads - 1) / kThreads;   // pieces per thread
  __shared__ __attribute__((aligned(16))) double2 sT[16 * NW * kCols];
  __shared__ __attribute__((aligned(16))) char sL[2][kCols * ROWB];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int w0 = blockIdx.x * Rw;
  const int nw = min(Rw, W - w0);                 // walkers of this workgroup
  const int nbeg = blockIdx.y * chunk, nend = min(K, nbeg + chunk);
  const int ns = (M + kKS - 1) / kKS;

  // ---- the wavefront's rows of G: lane (g, r16) holds row 16 wave + r16, k = KS c + SPS g + s
  double ar[NS][SPS], ai[NS][SPS];
  {
    const int row = 16 * wave + r16;
    const bool ok = row < nw * N;
    const double2* Gr = reinterpret_cast<const double2*>(G) + ((long)w0 * N + (ok ? row : 0)) * M;
#pragma unroll
    for (int c = 0; c < NS; ++c)
#pragma unroll
      for (int s = 0; s < SPS; ++s) {
        const int k = kKS * c + SPS * g + s;
        double2 x = double2{0.0, 0.0};
        if (ok && k < M) x = Gr[k];
        if (!LC) {
          const double bad = (x.x - x.x) + (x.y - x.y);   // 0, or NaN for a NaN or Inf
          x.x += bad;
          x.y += bad;
        }
        ar[c][s] = x.x;
        ai[c][s] = x.y;
      }
  }

  // ---- staging of the columns: piece p of the thread is 16 bytes of row p / TPR
  const long ncol = (long)K * N;
  uint4 pre[PCS];
  auto gload = [&](long col0, int c) {
#pragma unroll
    for (int i = 0; i < PCS; ++i) {
      const int p = tid + i * kThreads;
      const int row = p / TPR, q = p % TPR;
      const long col = min(col0 + row, ncol - 1);
      uint4 v = uint4{0u, 0u, 0u, 0u};
      if (PCS * kThreads == kCols * TPR || row < kCols) {
        if (LC) {
          const int k = kKS * c + q;
          if (k < M) v = *reinterpret_cast<const uint4*>(L + 2 * (col * M + k));
        } else {
          v = *reinterpret_cast<const uint4*>(L + col * ldl + kKS * c + 2 * q);
        }
      }
      pre[i] = v;
    }
  };
  auto lstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PCS; ++i) {
      const int p = tid + i * kThreads;
      const int row = p / TPR, q = p % TPR;
      if (PCS * kThreads == kCols * TPR || row < kCols)
        *reinterpret_cast<uint4*>(sL[buf] + row * ROWB + 16 * q) = pre[i];
    }
  };

  // ---- epilogue of one pass. Thread t of a walker takes the pairs (a, a + d mod N) of every
  // vector, d = 0 .. N/2: together each unordered pair once (twice with half the weight when
  // 2 d = N).
  const int tpw = kThreads / Rw;
  const int wl = tid / tpw, tl = tid - wl * tpw;
  const int D = N / 2 + 1;
  const int sa = tpw % N, sq = tpw / N, sd = sq % D, sv = sq / D;
  const int a0 = tl % N, d0 = (tl / N) % D, v0 = (tl / N) / D;
  const int gs = N <= 4 ? 4 : (N <= 8 ? 8 : 16);   // lanes per (walker, vector) trace
  double exx_re = 0.0, exx_im = 0.0;
  auto epilogue = [&](int n0) {
    const int nv = min(Cv, nend - n0);
    if (wl < nw) {
      const double2* T = sT + wl * N * kCols;
      for (int a = a0, d = d0, v = v0; v < nv;) {
        int b = a + d;
        if (b >= N) b -= N;
        const double2 x = T[a * kCols + v * N + b], y = T[b * kCols + v * N + a];
        const double wt = (d == 0 || 2 * d == N) ? 1.0 : 2.0;
        exx_re += wt * (x.x * y.x - x.y * y.y);
        exx_im += wt * (x.x * y.y + x.y * y.x);
        a += sa;
        d += sd;
        v += sv;
        if (a >= N) {
          a -= N;
          ++d;
        }
        if (d >= D) {
          d -= D;
          ++v;
        }
      }
    }
    const int np = nw * nv;
    for (int p0 = 0; p0 < np; p0 += kThreads / gs) {
      const int p = p0 + tid / gs;
      const int w = p / nv, v = p - w * nv;
      double dr = 0.0, di = 0.0;
      if (p < np)
        for (int a = tid & (gs - 1); a < N; a += gs) {
          const double2 x = sT[(w * N + a) * kCols + v * N + a];
          dr += x.x;
          di += x.y;
        }
      for (int off = gs >> 1; off > 0; off >>= 1) {
        dr += __shfl_xor(dr, off, 64);
        di += __shfl_xor(di, off, 64);
      }
      if (p < np && (tid & (gs - 1)) == 0)
        *reinterpret_cast<double2*>(Kl + 2 * ((long)(w0 + w) * K + n0 + v)) = double2{dr, di};
    }
  };

  if (nbeg < nend) {
    gload((long)nbeg * N, 0);
    lstore(0);
  }
  __syncthreads();
  int buf = 0;
  const int eslice = wave < NW / 2 ? 0 : ns / 2;   // slice of the last pass's epilogue
  for (int n0 = nbeg; n0 < nend; n0 += Cv) {
    d4 cr[CT], ci[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      cr[t] = d4{0, 0, 0, 0};
      ci[t] = d4{0, 0, 0, 0};
    }
#pragma unroll
    for (int c = 0; c < NS; ++c) {
      if (c < ns) {
        const bool last = c + 1 >= ns;
        const bool more = !last || n0 + Cv < nend;
        if (more) gload((long)(last ? n0 + Cv : n0) * N, last ? 0 : c + 1);
        if (c == eslice && n0 > nbeg) epilogue(n0 - Cv);
        const char* base = sL[buf] + r16 * ROWB + SPS * g * EB;
        if (LC) {
#pragma unroll
          for (int s = 0; s < SPS; ++s) {
            double br[CT], bi[CT];
#pragma unroll
            for (int t = 0; t < CT; ++t) {
              const double2 x = *reinterpret_cast<const double2*>(base + t * 16 * ROWB + s * 16);
              br[t] = x.x;
              bi[t] = x.y;
            }
#pragma unroll
            for (int t = 0; t < CT; ++t) {
              cr[t] = mfma16x16x4(ar[c][s], br[t], cr[t]);
              ci[t] = mfma16x16x4(ar[c][s], bi[t], ci[t]);
            }
#pragma unroll
            for (int t = 0; t < CT; ++t) {
              cr[t] = mfma16x16x4(-ai[c][s], bi[t], cr[t]);
              ci[t] = mfma16x16x4(ai[c][s], br[t], ci[t]);
            }
          }
        } else {
#pragma unroll
          for (int s = 0; s < SPS; s += 2) {
            double2 b[CT];
#pragma unroll
            for (int t = 0; t < CT; ++t)
              b[t] = *reinterpret_cast<const double2*>(base + t * 16 * ROWB + s * 8);
#pragma unroll
            for (int t = 0; t < CT; ++t) {
              cr[t] = mfma16x16x4(ar[c][s], b[t].x, cr[t]);
              ci[t] = mfma16x16x4(ai[c][s], b[t].x, ci[t]);
            }
#pragma unroll
            for (int t = 0; t < CT; ++t) {
              cr[t] = mfma16x16x4(ar[c][s + 1], b[t].y, cr[t]);
              ci[t] = mfma16x16x4(ai[c][s + 1], b[t].y, ci[t]);
            }
          }
        }
        // the other buffer was last read in the previous slice, before the barrier that ended it
        if (more) lstore(buf ^ 1);
        buf ^= 1;
        __syncthreads();
      }
    }
    // every wavefront has read the previous pass's T before the barrier of the last slice
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sT[(16 * wave + acc_row<double>(g, r)) * kCols + 16 * t + r16] =
            double2{cr[t][r], ci[t][r]};
    __syncthreads();
  }
  if (nbeg < nend) epilogue(nbeg + (nend - 1 - nbeg) / Cv * Cv);

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

struct Plan {
  int nw, ct, rw, cv, chunk, nchunk;   // wavefronts, column tiles, walkers, vectors per pass
};

// Column tiles: 3 (48 columns) where they hold the vectors with less padding than 4 (64 columns):
// N = 24 fills 3 tiles with 2 vectors and 3/4 of 4 tiles. Wavefronts: 8 (128 rows, two per SIMD),
// or 4 where workgroups of 8 would leave CUs without work. The vectors are split into chunks that
// minimise the rounds of workgroups times (passes + 1), the 1 standing for a workgroup's reading
// of G.
Plan plan_of(int W, int N, int K) {
  Plan p;
  const int c3 = 48 / N, c4 = 64 / N;
  p.ct = c3 * 64 > c4 * 48 ? 3 : 4;
  p.cv = std::min(p.ct == 3 ? c3 : c4, K);
  const long passes = (K + p.cv - 1) / p.cv;
  const long cus = device_cus();
  p.nw = ((long)(W + 128 / N - 1) / (128 / N)) * passes >= cus ? 8 : 4;
  p.rw = 16 * p.nw / N;
  const long groups = (W + p.rw - 1) / p.rw;
  long best = -1;
  p.chunk = K;
  for (long nch = 1; nch <= passes; ++nch) {
    const long per = (passes + nch - 1) / nch;
    const long cost = ((groups * ((passes + per - 1) / per) + cus - 1) / cus) * (per + 1);
    if (best < 0 || cost < best) {
      best = cost;
      p.chunk = (int)per * p.cv;
    }
  }
  p.nchunk = (K + p.chunk - 1) / p.chunk;
  return p;
}

}  // namespace

bool exchange_f64_supported(int M, int N) { return M <= 128 && N <= 32; }

int exchange_f64_chunks(int W, int N, int K) { return plan_of(W, N, K).nchunk; }

// Fitted to 996 measured calls (M 16 to 128, N 3 to 32, K 8 to 640, 1 to 1024 walkers): 90 % within 0.89 to
// 1.11 of the time. Per pass the tiles' MFMAs (two for complex vectors) and the pair sums, per round G.
double exchange_f64_us(int W, int M, int N, int K, bool real) {
  const Plan p = plan_of(W, N, K);
  const long wgs = (long)((W + p.rw - 1) / p.rw) * p.nchunk, cus = device_cus();
  const double rounds = (double)((wgs + cus - 1) / cus), passes = rounds * ((p.chunk + p.cv - 1) / p.cv);
  const double tiles = p.nw * p.ct * ((M + 15) / 16), g = p.nw * ((M + 15) / 16);
  return real ? 6.8 + passes * (0.064 * tiles + 3.6) + 0.17 * rounds * g
              : 6.6 + passes * (0.131 * tiles + 3.2) + 0.24 * rounds * g;
}

int real_lnak_row(int M) { return (M + 15) / 16 * 16; }

void launch_exchange_f64(hipStream_t s, int W, int M, int N, int K, const double* G,
                         const double* Lnak, const double* Lreal, double* Kl, double* part) {
  if (W <= 0 || K <= 0) return;
  AFQ_CHECK(exchange_f64_supported(M, N), AFQ_EUNSUPPORTED, "FP64 exchange: needs N <= 32, M <= 128");
  const Plan p = plan_of(W, N, K);
  const dim3 grid((W + p.rw - 1) / p.rw, p.nchunk);
  const double* L = Lreal ? Lreal : Lnak;
  const int ldl = real_lnak_row(M);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(64 * p.nw), 0, s, W, M, N, K, ldl, p.rw, p.cv, p.chunk, G,
                       L, Kl, part, p.nchunk);
  };
  auto pick = [&](auto kch) {
    constexpr int KCH = decltype(kch)::value;
    if (Lreal) {
      if (p.ct == 3) p.nw == 8 ? go(k_exchange_f64<KCH, 3, false, 8>) : go(k_exchange_f64<KCH, 3, false, 4>);
      else p.nw == 8 ? go(k_exchange_f64<KCH, 4, false, 8>) : go(k_exchange_f64<KCH, 4, false, 4>);
    } else {
      if (p.ct == 3) p.nw == 8 ? go(k_exchange_f64<KCH, 3, true, 8>) : go(k_exchange_f64<KCH, 3, true, 4>);
      else p.nw == 8 ? go(k_exchange_f64<KCH, 4, true, 8>) : go(k_exchange_f64<KCH, 4, true, 4>);
    }
  };
  if (M <= 32) pick(std::integral_constant<int, 2>());
  else if (M <= 64) pick(std::integral_constant<int, 4>());
  else if (M <= 96) pick(std::integral_constant<int, 6>());
  else pick(std::integral_constant<int, 8>());
  AFQ_HIP(hipGetLastError());
}

}  // namespace afq
