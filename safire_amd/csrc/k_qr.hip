// Batched re-orthogonalisation of walkers (det_ops::orthogonalize, orthogonalize.hpp:131-169):
// Householder QR of Phi_w [M,N] with LAPACK zgeqrf conventions (zlarfg: real
// beta = -sign(Re alpha) |x|, tau = (beta - alpha)/beta, v = x/(alpha - beta)), log det R
// accumulated as log_determinant_from_geqrf does (determinants_impl.hpp:77-108), Q formed by
// backward accumulation (zungqr), and Q's columns scaled by sign(Re R_ii): the result is the
// unique Q whose R has a positive real diagonal.
//
// k_qr_regs (M <= 128): 8 threads per column hold the column of A and then of Q in registers (rows
// q, q + 8, ...), one workgroup per walker. A step's reflector v goes through LDS once (double-
// buffered, one barrier per step): its 8 owners form it, every thread reads its rows of it, and
// a column's dot product takes three DPP additions over its 8 lanes. So the 2 N serial steps cost
// an LDS read of M / 8 entries, M / 4 complex multiply-adds and a short reduction each. M 128, N 32,
// 1024 walkers: 928 us with A and Q in LDS and a wavefront-wide shuffle reduction per column
// (k_qr, which stays for M > 128 and for few columns of more than 64 rows), 252 us here; M 48, N 12, 256
// walkers: 46 -> 22 us.
//
// k_qr: one workgroup per walker; A (the reflectors) and Q live in LDS with rows padded to N + 1
// complex numbers, so that the lanes of a column access (consecutive rows) fall into different
// banks instead of all into one. Each elimination step reduces a column norm in one wavefront and
// applies the reflector with one wavefront per trailing column (lanes over rows, shuffle
// reductions).
#include "afq_internal.hpp"

#include <cfloat>

namespace afq {

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

__device__ inline cd wave_sum(cd v) {
  for (int off = 32; off > 0; off >>= 1) {
    v.re += __shfl_xor(v.re, off, 64);
    v.im += __shfl_xor(v.im, off, 64);
  }
  return v;
}

__global__ __launch_bounds__(kThreads) void k_qr(int M, int N, cd* __restrict__ Phi, long ldw,
                                                 cd* __restrict__ logdetR) {
  extern __shared__ cd smem[];
  const int ld = N + 1;    // padded row stride
  cd* A = smem;            // [M][ld]
  cd* Q = A + M * ld;      // [M][ld]
  __shared__ cd tau[64];
  __shared__ double scl[64];
  const int w = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  cd* P = Phi + (long)w * ldw;
  for (int e = tid; e < M * N; e += kThreads) A[(e / N) * ld + e % N] = P[e];
  __syncthreads();
  const int kmax = min(M, N);

  for (int j = 0; j < kmax; ++j) {
    if (wave == 0) {
      double x2 = 0.0;
      for (int i = j + 1 + lane; i < M; i += 64) x2 += cnorm(A[i * ld + j]);
      for (int off = 32; off > 0; off >>= 1) x2 += __shfl_xor(x2, off, 64);
      const cd alpha = A[j * ld + j];
      cd t = cmk(0.0, 0.0), sc = cmk(0.0, 0.0);
      double beta = 0.0;
      const bool identity = (x2 == 0.0 && alpha.im == 0.0);
      if (!identity) {
        const double nrm = sqrt(cnorm(alpha) + x2);
        beta = (alpha.re >= 0.0) ? -nrm : nrm;
        t = cmk((beta - alpha.re) / beta, -alpha.im / beta);
        sc = cdiv(cmk(1.0, 0.0), cmk(alpha.re - beta, alpha.im));
      }
      for (int i = j + 1 + lane; i < M; i += 64)
        if (!identity) A[i * ld + j] = A[i * ld + j] * sc;
      if (lane == 0) {
        tau[j] = t;
        if (!identity) A[j * ld + j] = cmk(beta, 0.0);
      }
    }
    __syncthreads();
    // A[j:, c] -= conj(tau) v (v^H A[j:, c]) for c > j
    const cd tj = cconj(tau[j]);
    for (int c = j + 1 + wave; c < N; c += kWaves) {
      cd s = cmk(0.0, 0.0);
      for (int i = j + 1 + lane; i < M; i += 64) s += cconj(A[i * ld + j]) * A[i * ld + c];
      s = wave_sum(s);
      s = (A[j * ld + c] + s);
      s = tj * s;
      if (lane == 0) A[j * ld + c] -= s;
      for (int i = j + 1 + lane; i < M; i += 64) A[i * ld + c] -= s * A[i * ld + j];
    }
    __syncthreads();
  }

  if (tid < kmax) scl[tid] = (A[tid * ld + tid].re < 0.0) ? -1.0 : 1.0;
  if (logdetR != nullptr && tid == 0) {
    cd acc = logdetR[w];
    for (int i = 0; i < kmax; ++i) {
      const cd r = (A[i * ld + i].re < 0.0) ? -A[i * ld + i] : A[i * ld + i];
      acc += clog_(cmk(r.re + DBL_MIN, r.im));
    }
    logdetR[w] = acc;
  }
  for (int e = tid; e < M * N; e += kThreads) {
    const int i = e / N, c = e - i * N;
    Q[i * ld + c] = cmk(i == c ? 1.0 : 0.0, 0.0);
  }
  __syncthreads();
  for (int j = kmax - 1; j >= 0; --j) {
    const cd t = tau[j];
    for (int c = j + wave; c < N; c += kWaves) {
      cd s = cmk(0.0, 0.0);
      for (int i = j + 1 + lane; i < M; i += 64) s += cconj(A[i * ld + j]) * Q[i * ld + c];
      s = wave_sum(s);
      s = t * (Q[j * ld + c] + s);
      if (lane == 0) Q[j * ld + c] -= s;
      for (int i = j + 1 + lane; i < M; i += 64) Q[i * ld + c] -= s * A[i * ld + j];
    }
    __syncthreads();
  }
  for (int e = tid; e < M * N; e += kThreads) {
    const int i = e / N, c = e % N;
    P[e] = (c < kmax) ? scl[c] * Q[i * ld + c] : Q[i * ld + c];
  }
}

template <int CTRL>
__device__ inline double dpp_add(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_update_dpp((unsigned)u, (unsigned)u, CTRL, 0xf, 0xf, false);
  const unsigned hi = __builtin_amdgcn_update_dpp((unsigned)(u >> 32), (unsigned)(u >> 32), CTRL, 0xf,
                                                  0xf, false);
  return v + __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// the sum over the 8 lanes of a column, in all of them: lanes ^1, ^2 (quad permutes), then the other
// quad (mirror of the half row)
__device__ inline double sum8(double v) {
  v = dpp_add<0xB1>(v);
  v = dpp_add<0x4E>(v);
  return dpp_add<0x141>(v);
}

template <int RPT>
__global__ __launch_bounds__(512) void k_qr_regs(int M, int N, cd* __restrict__ Phi, long ldw,
                                                 cd* __restrict__ logdetR) {
  __shared__ cd sV[2][8 * RPT];
  __shared__ cd sTau[64];
  __shared__ cd sR[64];            // diagonal of R
  const int w = blockIdx.x, tid = threadIdx.x;
  const int c = tid >> 3, q = tid & 7;
  const int cmax = __builtin_amdgcn_readfirstlane((tid & ~63) >> 3) + 7;   // the wavefront's last column
  cd* P = Phi + (long)w * ldw;
  cd a[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = q + 8 * i;
    a[i] = (c < N && r < M) ? P[(long)r * N + c] : cmk(0.0, 0.0);
  }
  // reflector of column j by its owners: v (0 above row j, 1 in it) to LDS, and below row j into a[]
  auto reflector = [&](int j) {
    double x2 = 0.0;
    cd al = cmk(0.0, 0.0);
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = q + 8 * i;
      if (r > j) x2 += cnorm(a[i]);
      if (r == j) al = a[i];
    }
    x2 = sum8(x2);
    al.re = sum8(al.re);
    al.im = sum8(al.im);
    cd t = cmk(0.0, 0.0), sc = cmk(1.0, 0.0), diag = al;
    if (!(x2 == 0.0 && al.im == 0.0)) {
      const double nrm = sqrt(cnorm(al) + x2);
      const double beta = (al.re >= 0.0) ? -nrm : nrm;
      t = cmk((beta - al.re) / beta, -al.im / beta);
      sc = cdiv(cmk(1.0, 0.0), cmk(al.re - beta, al.im));
      diag = cmk(beta, 0.0);
    }
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = q + 8 * i;
      if (r > j) a[i] = a[i] * sc;
      sV[j & 1][r] = r > j ? a[i] : cmk(r == j ? 1.0 : 0.0, 0.0);
    }
    if (q == 0) {
      sTau[j] = t;
      sR[j] = diag;
    }
  };
  // x -= t (v^H x) v
  auto apply = [&](cd (&x)[RPT], const cd* v, cd t) {
    cd s = cmk(0.0, 0.0), vi[RPT];
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      vi[i] = v[q + 8 * i];
      s += cconj(vi[i]) * x[i];
    }
    s.re = sum8(s.re);
    s.im = sum8(s.im);
    s = t * s;
#pragma unroll
    for (int i = 0; i < RPT; ++i) x[i] -= s * vi[i];
  };

  if (c == 0) reflector(0);
  __syncthreads();
  for (int j = 0; j < N; ++j) {
    if (cmax > j) {
      if (c > j && c < N) apply(a, sV[j & 1], cconj(sTau[j]));
      if (c == j + 1 && c < N) reflector(j + 1);   // into the other buffer
    }
    __syncthreads();
  }
  if (logdetR != nullptr && tid < 64) {
    cd acc = cmk(0.0, 0.0);
    if (tid < N) {
      const cd r = (sR[tid].re < 0.0) ? -sR[tid] : sR[tid];
      acc = clog_(cmk(r.re + DBL_MIN, r.im));
    }
    acc = wave_sum(acc);
    if (tid == 0) logdetR[w] += acc;
  }
  // Q by backward accumulation, H_1 .. H_N applied to the identity
  cd x[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) x[i] = cmk(q + 8 * i == c ? 1.0 : 0.0, 0.0);
  for (int j = N - 1; j >= 0; --j) {
    if (c == j)
#pragma unroll
      for (int i = 0; i < RPT; ++i) {
        const int r = q + 8 * i;
        sV[j & 1][r] = r > j ? a[i] : cmk(r == j ? 1.0 : 0.0, 0.0);
      }
    __syncthreads();
    if (cmax >= j && c >= j && c < N) apply(x, sV[j & 1], sTau[j]);
  }
  if (c < N) {
    const double scl = (sR[c].re < 0.0) ? -1.0 : 1.0;
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = q + 8 * i;
      if (r < M) P[(long)r * N + c] = scl * x[i];
    }
  }
}

}  // namespace

void launch_orthogonalize(hipStream_t s, int nb, int M, int N, double* Phi, long ldw,
                          double* logdetR) {
  if (nb <= 0 || (long)M * N == 0) return;
  AFQ_CHECK(N <= 64, AFQ_EUNSUPPORTED, "orthogonalize: N > 64");
  const size_t lds = 2 * sizeof(cd) * (size_t)M * (N + 1);
  AFQ_CHECK(lds <= 160 * 1024 - 2048, AFQ_EUNSUPPORTED, "orthogonalize: walker too large");
  // Up to four columns leave the 8 threads of each with all of its rows, one after the other: k_qr is
  // faster (us, k_qr and k_qr_regs at 256 walkers: M 128, N 2 8.7 and 11.4, N 3 13.1 and 14.6, N 4 14.9
  // and 18.1, N 5 20.1 and 20.4; M 65, N 2 8.2 and 9.1, N 4 13.4 and 14.5; M 96, N 3 12.6 and 12.0; M 64,
  // N 2 both 8) until more walkers share a CU (M 128, N 2: 1024 10.1 and 13.1, 2048 18.5 and 16.0; N 4:
  // 512 17.0 and 19.3, 1024 20.8 and 19.6)
  const int cus = device_cus();
  const bool few = M > 64 && (N <= 2 ? nb <= 4 * cus : N <= 4 && (M > 96 ? nb <= 2 * cus : N == 4 && nb <= cus));
  if (M <= 128 && N <= M && !few) {
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(nb), dim3((8 * N + 63) / 64 * 64), 0, s, M, N,
                         reinterpret_cast<cd*>(Phi), ldw, reinterpret_cast<cd*>(logdetR));
    };
    if (M <= 16) go(k_qr_regs<2>);
    else if (M <= 32) go(k_qr_regs<4>);
    else if (M <= 48) go(k_qr_regs<6>);
    else if (M <= 64) go(k_qr_regs<8>);
    else if (M <= 96) go(k_qr_regs<12>);
    else go(k_qr_regs<16>);
    AFQ_HIP(hipGetLastError());
    return;
  }
  ensure_dynamic_lds((const void*)k_qr, lds);
  hipLaunchKernelGGL(k_qr, dim3(nb), dim3(kThreads), lds, s, M, N, reinterpret_cast<cd*>(Phi),
                     ldw, reinterpret_cast<cd*>(logdetR));
  AFQ_HIP(hipGetLastError());
}

}  // namespace afq
