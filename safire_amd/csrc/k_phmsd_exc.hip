// Energy and density matrix of a particle-hole expansion from rank-nex corrections of the reference
// determinant (PHMSD::energy_alg1, PHMSD.cpp:377-544; PHMSD::MixedDensityMatrix, 549-795).
//
// With T^n[i][a] = sum_k G[i][k] Lna[n][a][k] of the reference's compact G (the reference occupies
// orbitals 0..nel-1, columns i < nel of T^n are its exchange block), QQ0[a][i] the projection of
// orbital a on the reference, and for determinant d (holes p_1..p_r to particles v_1..v_r)
// Q = A^-1, A(p, q) = QQ0[v_p][p_q], the determinant's exchange block is the reference's with r
// changed columns:
//
//   X_d[i][p_e] = T[i][p_e] + sum_q Q(e, q) S[i][v_q],    S[i][v] = T[i][v] - sum_j T[i][j] QQ0[v][j]
//
// (the sums over all occupied columns that the compact R matrices carry are taken once per vector,
// in S). So with B[p][v] = sum_j T[p][j] S[j][v] and D(f, q) = S[p_f][v_q], M = D Q^T:
//
//   tr X_d  = tr T + tr M,    tr X_d^2 = tr T^2 + 2 sum_eq Q(e, q) B[p_e][v_q] + tr M^2
//
// r^3 + 2 r^2 complex multiply-adds per determinant and vector instead of nel nact r: 24 instead of
// 1408 for doubles in 64 orbitals. A workgroup takes a walker and NV vectors, forms S and B for
// its particle columns in LDS, and sweeps all determinants with a thread per determinant, whose Q
// is read once for the NV vectors. The one-body matrix rides along as vector nchol (only the trace
// change is used there). Bound by LDS gathers and FP64 VALU work. 64 orbitals, 10 + 10 electrons,
// 320 vectors, 1000 determinants, 256 walkers: the energy 266 -> 6.8 ms against the kernels that
// apply the compact R (k_ph_2body_lds; they stay for S and B that do not fit LDS and for callers
// that bring their own R), the force bias 19.4 -> 2.0 ms. The up spin writes its traces KE[w][n][u], determinants fastest; the down
// spin picks them up through the CI couplings. Fixed-order sums throughout.
//
#include "afq_internal.hpp"

#include <algorithm>

namespace afq {

namespace {

constexpr int kThreads = 256;

__device__ inline cd wsum(cd v) {
  for (int off = 32; off > 0; off >>= 1) {
    v.re += __shfl_xor(v.re, off, 64);
    v.im += __shfl_xor(v.im, off, 64);
  }
  return v;
}

// det and inverse of a NEX x NEX matrix by Gauss-Jordan with partial pivoting (first maximum of
// |re| + |im|); false when a pivot is exactly zero
template <int NEX>
__device__ inline bool invert(cd (&a)[NEX][NEX], cd (&q)[NEX][NEX], cd& det) {
#pragma unroll
  for (int i = 0; i < NEX; ++i)
#pragma unroll
    for (int j = 0; j < NEX; ++j) q[i][j] = cmk(i == j ? 1.0 : 0.0, 0.0);
  det = cmk(1.0, 0.0);
#pragma unroll
  for (int j = 0; j < NEX; ++j) {
    int p = j;
    double best = cabs1(a[j][j]);
#pragma unroll
    for (int r = j + 1; r < NEX; ++r)
      if (cabs1(a[r][j]) > best) {
        best = cabs1(a[r][j]);
        p = r;
      }
    if (p != j) {
      det = -det;
#pragma unroll
      for (int r = j + 1; r < NEX; ++r)
        if (r == p)
#pragma unroll
          for (int c = 0; c < NEX; ++c) {
            const cd t = a[j][c];
            a[j][c] = a[r][c];
            a[r][c] = t;
            const cd u = q[j][c];
            q[j][c] = q[r][c];
            q[r][c] = u;
          }
    }
    const cd piv = a[j][j];
    det = det * piv;
    if (cis0(piv)) return false;
    const cd inv = cdiv(cmk(1.0, 0.0), piv);
#pragma unroll
    for (int c = 0; c < NEX; ++c) {
      a[j][c] = a[j][c] * inv;
      q[j][c] = q[j][c] * inv;
    }
#pragma unroll
    for (int r = 0; r < NEX; ++r) {
      if (r == j) continue;
      const cd f = a[r][j];
#pragma unroll
      for (int c = 0; c < NEX; ++c) {
        a[r][c] -= f * a[j][c];
        q[r][c] -= f * q[j][c];
      }
    }
  }
  return true;
}

// the overlap ratio and Q of determinant d of a shell: Q[w][qoff + eq ndet + d], ratio[row + d][w]
template <int NEX>
__device__ inline void one_ratio(const PhShell& sh, int nw, int nel, int w, int d,
                                 const cd* __restrict__ QQ0w, cd* __restrict__ ratio,
                                 cd* __restrict__ Qw) {
  const int* e = sh.iexcit + (long)d * 2 * NEX;
  cd a[NEX][NEX], q[NEX][NEX], det;
#pragma unroll
  for (int r = 0; r < NEX; ++r)
#pragma unroll
    for (int c = 0; c < NEX; ++c) a[r][c] = QQ0w[(long)e[NEX + r] * nel + e[c]];
  const bool ok = invert<NEX>(a, q, det);
  ratio[(long)(sh.row + d) * nw + w] = ok ? det : cmk(0.0, 0.0);
#pragma unroll
  for (int r = 0; r < NEX; ++r)
#pragma unroll
    for (int c = 0; c < NEX; ++c)
      Qw[sh.qoff + (long)(r * NEX + c) * sh.ndet + d] = ok ? q[r][c] : cmk(0.0, 0.0);
}

template <int MAXNEX>
__global__ __launch_bounds__(kThreads) void k_ph_ratios_q(int nw, int nel, int nact, long qtot,
                                                          const PhShell* __restrict__ shells,
                                                          const cd* __restrict__ QQ0,
                                                          cd* __restrict__ ratio,
                                                          cd* __restrict__ Q) {
  const PhShell sh = shells[blockIdx.y];
  const long id = (long)blockIdx.x * kThreads + threadIdx.x;
  if (blockIdx.y == 0 && id < nw) ratio[id] = cmk(1.0, 0.0);   // the reference
  if (id >= (long)sh.ndet * nw) return;
  const int w = (int)(id / sh.ndet), d = (int)(id % sh.ndet);
  const cd* T = QQ0 + (long)w * nact * nel;
  cd* Qw = Q + w * qtot;
  switch (sh.nex) {
    case 1: one_ratio<1>(sh, nw, nel, w, d, T, ratio, Qw); break;
    case 2: one_ratio<2>(sh, nw, nel, w, d, T, ratio, Qw); break;
    case 3: one_ratio<3>(sh, nw, nel, w, d, T, ratio, Qw); break;
    case 4: one_ratio<4>(sh, nw, nel, w, d, T, ratio, Qw); break;
    default:
      if constexpr (MAXNEX > 4) {
        switch (sh.nex) {
          case 5: one_ratio<5>(sh, nw, nel, w, d, T, ratio, Qw); break;
          case 6: one_ratio<6>(sh, nw, nel, w, d, T, ratio, Qw); break;
          case 7: one_ratio<7>(sh, nw, nel, w, d, T, ratio, Qw); break;
          default: one_ratio<8>(sh, nw, nel, w, d, T, ratio, Qw); break;
        }
      }
  }
}

// wgt[u][w] = own[u][w] sum_{d in row u} C[u][d] other[d][w] (PHMSD.cpp:441-450): a workgroup per row
// and 32 walkers, 8 threads of a walker sharing the row's entries (the reference's row couples to
// every determinant that excites the other spin only)
__global__ __launch_bounds__(256) void k_ph_weights(int nw, const int* __restrict__ cp,
                                                    const int* __restrict__ ci,
                                                    const cd* __restrict__ cv,
                                                    const cd* __restrict__ own,
                                                    const cd* __restrict__ other,
                                                    cd* __restrict__ wgt) {
  __shared__ cd part[8][32];
  const int u = blockIdx.x, wl = threadIdx.x & 31, jl = threadIdx.x >> 5;
  const int w = blockIdx.y * 32 + wl;
  const int j0 = cp[u], j1 = cp[u + 1];
  cd acc = cmk(0.0, 0.0);
  if (w < nw)
    for (int j = j0 + jl; j < j1; j += 8) acc += cv[j] * other[(long)ci[j] * nw + w];
  part[jl][wl] = acc;
  __syncthreads();
  if (jl == 0 && w < nw) {
    for (int q = 1; q < 8; ++q) acc += part[q][wl];
    wgt[(long)u * nw + w] = acc * own[(long)u * nw + w];
  }
}

// out[w] = sum_u wgt[u][w]; one wavefront per walker
__global__ __launch_bounds__(64) void k_ph_weight_sum(int nw, int nu, const cd* __restrict__ wgt,
                                                      cd* __restrict__ out) {
  const int w = blockIdx.x;
  cd acc = cmk(0.0, 0.0);
  for (int u = threadIdx.x; u < nu; u += 64) acc += wgt[(long)u * nw + w];
  acc = wsum(acc);
  if (threadIdx.x == 0) out[w] = acc;
}

struct ExcSums {
  cd ex, ej, e1, cross;
};

// all determinants of one shell against the NV vectors of the workgroup
template <int NEX, int NV, bool DOWN>
__device__ inline void shell_sums(const PhShell& sh, int w, int nw, int nel, int nvir, int nchol,
                                  int n0, int nu_own, int nu_up, const cd* __restrict__ Qw,
                                  const cd* __restrict__ wgt, const cd* sS, const cd* sB,
                                  const cd* sK0, cd* __restrict__ KEw, const int* __restrict__ cp,
                                  const int* __restrict__ ci, const cd* __restrict__ cv,
                                  const cd* __restrict__ rup, const cd* __restrict__ rdn,
                                  ExcSums& sum) {
  const int per = nel * nvir;
  for (int d = threadIdx.x; d < sh.ndet; d += kThreads) {
    const int* ex = sh.iexcit + (long)d * 2 * NEX;
    int p[NEX], v[NEX];
    cd q[NEX][NEX];
#pragma unroll
    for (int e = 0; e < NEX; ++e) {
      p[e] = ex[e] * nvir;
      v[e] = ex[NEX + e] - nel;
    }
#pragma unroll
    for (int e = 0; e < NEX; ++e)
#pragma unroll
      for (int f = 0; f < NEX; ++f) q[e][f] = Qw[sh.qoff + (long)(e * NEX + f) * sh.ndet + d];
    const int u = sh.row + d;
    const cd wd = wgt[(long)u * nw + w];
    cd kn[NV];
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      kn[n] = cmk(0.0, 0.0);
      if (n0 + n > nchol) continue;
      const cd* S = sS + n * per;
      const cd* B = sB + n * per;
      cd m[NEX][NEX], b = cmk(0.0, 0.0), tr = cmk(0.0, 0.0);
#pragma unroll
      for (int f = 0; f < NEX; ++f) {
        cd s[NEX];
#pragma unroll
        for (int k = 0; k < NEX; ++k) s[k] = S[p[f] + v[k]];
#pragma unroll
        for (int e = 0; e < NEX; ++e) {
          cd x = cmk(0.0, 0.0);
#pragma unroll
          for (int k = 0; k < NEX; ++k) x += s[k] * q[e][k];
          m[f][e] = x;
        }
        tr += m[f][f];
      }
      if (n0 + n == nchol) {   // the one-body matrix
        sum.e1 += wd * tr;
        continue;
      }
#pragma unroll
      for (int e = 0; e < NEX; ++e)
#pragma unroll
        for (int k = 0; k < NEX; ++k) b += q[e][k] * B[p[e] + v[k]];
      cd t2 = cmk(0.0, 0.0);
#pragma unroll
      for (int e = 0; e < NEX; ++e) {
        t2 += m[e][e] * m[e][e];
#pragma unroll
        for (int f = e + 1; f < NEX; ++f) t2 += 2.0 * (m[f][e] * m[e][f]);
      }
      const cd k0 = sK0[n];
      kn[n] = k0 + tr;
      sum.ex += wd * (2.0 * b + t2);
      // kn^2 - k0^2 = (kn + k0) tr
      sum.ej += wd * ((kn[n] + k0) * tr);
      if (!DOWN) KEw[(long)(n0 + n) * nu_own + u] = kn[n];
    }
    if (DOWN) {
      const cd rd = rdn[(long)u * nw + w];
      for (int j = cp[u]; j < cp[u + 1]; ++j) {
        const int c = ci[j];
        const cd coef = (cv[j] * rup[(long)c * nw + w]) * rd;
#pragma unroll
        for (int n = 0; n < NV; ++n)
          if (n0 + n < nchol) sum.cross += (coef * KEw[(long)(n0 + n) * nu_up + c]) * kn[n];
      }
    }
  }
}

// One walker, NV vectors, one spin. part[w][group][8]: ex, ej, e1, cross, tr T^2, (tr T)^2, tr of the
// one-body matrix.
template <int MAXNEX, int NV, bool DOWN>
__global__ __launch_bounds__(kThreads, 2) void k_ph_exc(
    int nw, int nel, int nact, int nchol, long qtot, int nshell, int nu_own, int nu_up,
    const PhShell* __restrict__ shells, const cd* __restrict__ T, const cd* __restrict__ QQ0,
    const cd* __restrict__ Q, const cd* __restrict__ wgt, cd* __restrict__ KE,
    const int* __restrict__ cp, const int* __restrict__ ci, const cd* __restrict__ cv,
    const cd* __restrict__ rup, const cd* __restrict__ rdn, cd* __restrict__ part) {
  extern __shared__ cd smem[];
  __shared__ cd sK0[NV], sX0[NV], red[kThreads / 64][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int w = blockIdx.x, n0 = blockIdx.y * NV;
  const int nvir = nact - nel, per = nel * nvir;
  cd* sT = smem;                    // [NV][nel][nel]
  cd* sS = sT + NV * nel * nel;     // [NV][nel][nvir]
  cd* sB = sS + NV * per;           // [NV][nel][nvir]
  const cd* Tw = T + (long)w * nel * (nchol + 1) * nact;
  auto Tat = [&](int i, int n, int a) -> cd {   // vectors past the one-body matrix: not used
    return Tw[((long)i * (nchol + 1) + min(n0 + n, nchol)) * nact + a];
  };
  for (int e = tid; e < NV * nel * nel; e += kThreads) {
    const int n = e / (nel * nel), r = e - n * nel * nel;
    sT[e] = Tat(r / nel, n, r % nel);
  }
  __syncthreads();
  // S and B, one particle column per thread; 8 rows at a time in registers
  for (int c = tid; c < NV * nvir; c += kThreads) {
    const int n = c / nvir, v = c - n * nvir;
    const cd* q = QQ0 + ((long)w * nact + nel + v) * nel;
    const cd* Tn = sT + n * nel * nel;
    cd* S = sS + n * per + v;
    cd* B = sB + n * per + v;
    for (int j0 = 0; j0 < nel; j0 += 8) {
      cd s[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) s[j] = Tat(min(j0 + j, nel - 1), n, nel + v);
      for (int i = 0; i < nel; ++i) {
        const cd qi = q[i];
#pragma unroll
        for (int j = 0; j < 8; ++j) s[j] -= Tn[min(j0 + j, nel - 1) * nel + i] * qi;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j0 + j < nel) S[(j0 + j) * nvir] = s[j];
    }
    for (int j0 = 0; j0 < nel; j0 += 8) {
      cd b[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) b[j] = cmk(0.0, 0.0);
      for (int i = 0; i < nel; ++i) {
        const cd si = S[i * nvir];
#pragma unroll
        for (int j = 0; j < 8; ++j) b[j] += Tn[min(j0 + j, nel - 1) * nel + i] * si;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j0 + j < nel) B[(j0 + j) * nvir] = b[j];
    }
  }
  // tr T and tr T^2 of the reference, a wavefront per vector
  for (int n = wave; n < NV; n += kThreads / 64) {
    const cd* Tn = sT + n * nel * nel;
    cd k = cmk(0.0, 0.0), x = cmk(0.0, 0.0);
    for (int e = lane; e < nel * nel; e += 64) {
      const int i = e / nel, j = e - i * nel;
      x += Tn[e] * Tn[j * nel + i];
      if (i == j) k += Tn[e];
    }
    k = wsum(k);
    x = wsum(x);
    if (lane == 0) {
      sK0[n] = k;
      sX0[n] = x;
    }
  }
  __syncthreads();
  ExcSums sum{cmk(0, 0), cmk(0, 0), cmk(0, 0), cmk(0, 0)};
  const cd* Qw = Q + w * qtot;
  cd* KEw = KE + (long)w * nchol * (DOWN ? nu_up : nu_own);
  // the reference's own row
  if (DOWN) {
    const cd rd = rdn[w];
    for (int j = cp[0] + tid; j < cp[1]; j += kThreads) {
      const int c = ci[j];
      const cd coef = (cv[j] * rup[(long)c * nw + w]) * rd;
#pragma unroll
      for (int n = 0; n < NV; ++n)
        if (n0 + n < nchol) sum.cross += (coef * KEw[(long)(n0 + n) * nu_up + c]) * sK0[n];
    }
  } else if (tid < NV && n0 + tid < nchol) {
    KEw[(long)(n0 + tid) * nu_own] = sK0[tid];
  }
  for (int h = 0; h < nshell; ++h) {
    const PhShell sh = shells[h];
    auto go = [&](auto nex) {
      shell_sums<decltype(nex)::value, NV, DOWN>(sh, w, nw, nel, nvir, nchol, n0, nu_own, nu_up, Qw,
                                                 wgt, sS, sB, sK0, KEw, cp, ci, cv, rup, rdn, sum);
    };
    switch (sh.nex) {
      case 1: go(std::integral_constant<int, 1>()); break;
      case 2: go(std::integral_constant<int, 2>()); break;
      case 3: go(std::integral_constant<int, 3>()); break;
      case 4: go(std::integral_constant<int, 4>()); break;
      default:
        if constexpr (MAXNEX > 4) {
          switch (sh.nex) {
            case 5: go(std::integral_constant<int, 5>()); break;
            case 6: go(std::integral_constant<int, 6>()); break;
            case 7: go(std::integral_constant<int, 7>()); break;
            default: go(std::integral_constant<int, 8>()); break;
          }
        }
    }
  }
  cd s[4] = {wsum(sum.ex), wsum(sum.ej), wsum(sum.e1), wsum(sum.cross)};
  if (lane == 0)
    for (int k = 0; k < 4; ++k) red[wave][k] = s[k];
  __syncthreads();
  cd* out = part + 8 * ((long)w * gridDim.y + blockIdx.y);
  if (tid < 4) {
    cd t = cmk(0.0, 0.0);
    for (int k = 0; k < kThreads / 64; ++k) t += red[k][tid];
    out[tid] = t;
  } else if (tid == 4) {
    cd x = cmk(0, 0), k2 = cmk(0, 0), h = cmk(0, 0);
    for (int n = 0; n < NV; ++n) {
      if (n0 + n < nchol) {
        x += sX0[n];
        k2 += sK0[n] * sK0[n];
      } else if (n0 + n == nchol) {
        h = sK0[n];
      }
    }
    out[4] = x;
    out[5] = k2;
    out[6] = h;
  }
}

// E[w] and the log overlap from the group sums of both spins and the weights (PHMSD.cpp:453-543); one
// wavefront per walker
__global__ __launch_bounds__(64) void k_ph_exc_finish(int nw, int nu, int gu, int gd, cd E0,
                                                      const cd* __restrict__ wgt,
                                                      const cd* __restrict__ pu,
                                                      const cd* __restrict__ pd,
                                                      const cd* __restrict__ log_ov,
                                                      cd* __restrict__ E, cd* __restrict__ ov) {
  const int w = blockIdx.x, lane = threadIdx.x;
  cd o = cmk(0, 0), s[2][7];
  for (int k = 0; k < 7; ++k) s[0][k] = s[1][k] = cmk(0, 0);
  for (int u = lane; u < nu; u += 64) o += wgt[(long)u * nw + w];
  for (int g = lane; g < gu; g += 64)
    for (int k = 0; k < 7; ++k) s[0][k] += pu[8 * ((long)w * gu + g) + k];
  for (int g = lane; g < gd; g += 64)
    for (int k = 0; k < 7; ++k) s[1][k] += pd[8 * ((long)w * gd + g) + k];
  o = wsum(o);
  for (int k = 0; k < 7; ++k) {
    s[0][k] = wsum(s[0][k]);
    s[1][k] = wsum(s[1][k]);
  }
  if (lane != 0) return;
  cd e[3] = {E0 * o, cmk(0, 0), cmk(0, 0)};
  for (int sp = 0; sp < 2; ++sp) {
    e[0] += s[sp][6] * o + s[sp][2];
    e[1] -= 0.5 * (s[sp][4] * o + s[sp][0]);
    e[2] += 0.5 * (s[sp][5] * o + s[sp][1]);
  }
  e[2] += s[1][3];
  for (int c = 0; c < 3; ++c) E[3L * w + c] = cdiv(e[c], o);
  ov[w] = clog_(o) + log_ov[w];
}

// R[w][i][a] of the whole expansion (calculate_R, phmsd_helpers.hpp:200-262): with
// Wm[p][v] = sum of wgt_d Q_d(e, q) over the determinants and (e, q) that excite p = p_e with
// particle v = v_q (listed per (p, v) in CSR form, in determinant order),
//   R[p][v] = Wm[p][v],   R[p][j] = delta(p, j) sum_d wgt_d - sum_v Wm[p][v] QQ0[v][j]  (j < nel)
// One workgroup per walker; ov[w] = sum_d wgt_d.
__global__ __launch_bounds__(kThreads) void k_ph_expansion_R(
    int nw, int nel, int nact, int nu, long qtot, const int* __restrict__ rp,
    const int* __restrict__ ru, const int* __restrict__ rq, const cd* __restrict__ QQ0,
    const cd* __restrict__ Q, const cd* __restrict__ wgt, cd* __restrict__ R,
    cd* __restrict__ ov) {
  __shared__ cd red[kThreads / 64];
  const int w = blockIdx.x, tid = threadIdx.x;
  const int nvir = nact - nel;
  cd* Rw = R + (long)w * nel * nact;
  const cd* Qw = Q + w * qtot;
  const cd* Pw = QQ0 + (long)w * nact * nel;
  cd o = cmk(0, 0);
  for (int u = tid; u < nu; u += kThreads) o += wgt[(long)u * nw + w];
  o = wsum(o);
  if ((tid & 63) == 0) red[tid >> 6] = o;
  for (int e = tid; e < nel * nvir; e += kThreads) {
    cd acc = cmk(0.0, 0.0);
    for (int j = rp[e]; j < rp[e + 1]; ++j) acc += wgt[(long)ru[j] * nw + w] * Qw[rq[j]];
    const int p = e / nvir, v = e - p * nvir;
    Rw[(long)p * nact + nel + v] = acc;
  }
  __syncthreads();   // the workgroup's own global writes are visible to it after the barrier
  o = cmk(0.0, 0.0);
  for (int k = 0; k < kThreads / 64; ++k) o += red[k];
  for (int e = tid; e < nel * nel; e += kThreads) {
    const int p = e / nel, j = e - p * nel;
    cd acc = p == j ? o : cmk(0.0, 0.0);
    for (int v = 0; v < nvir; ++v)
      acc -= Rw[(long)p * nact + nel + v] * Pw[(long)(nel + v) * nel + j];
    Rw[(long)p * nact + j] = acc;
  }
  if (tid == 0) ov[w] = o;
}

// U[w][i][l] = sum_a R[w][i][a] A[a][l]
__global__ __launch_bounds__(256) void k_ph_ra(int nel, int nact, int nmo,
                                               const cd* __restrict__ R, const cd* __restrict__ A,
                                               cd* __restrict__ U) {
  const int e = blockIdx.x * 256 + threadIdx.x, w = blockIdx.y;
  if (e >= nel * nmo) return;
  const int i = e / nmo, l = e - i * nmo;
  const cd* Rw = R + ((long)w * nel + i) * nact;
  cd acc = cmk(0.0, 0.0);
  for (int a = 0; a < nact; ++a) acc += Rw[a] * A[(long)a * nmo + l];
  U[((long)w * nel + i) * nmo + l] = acc;
}

// The spin-summed density in the orbital basis, F[w] = sum_s sum_i U_s[i][l] G_s[i][k] / ov[w]:
// folded, entry l <= k holding (l, k) + (k, l), for symmetric Cholesky vectors, or all nmo^2 entries
__global__ __launch_bounds__(256) void k_ph_density(int nup, int ndn, int nmo, int fold,
                                                    const cd* __restrict__ U0,
                                                    const cd* __restrict__ G0,
                                                    const cd* __restrict__ U1,
                                                    const cd* __restrict__ G1,
                                                    const cd* __restrict__ ov,
                                                    cd* __restrict__ F) {
  const int w = blockIdx.y, l = blockIdx.x;
  const cd* u0 = U0 + (long)w * nup * nmo;
  const cd* g0 = G0 + (long)w * nup * nmo;
  const cd* u1 = U1 + (long)w * ndn * nmo;
  const cd* g1 = G1 + (long)w * ndn * nmo;
  const cd inv = cdiv(cmk(1.0, 0.0), ov[w]);
  const int size = fold ? nmo * (nmo + 1) / 2 : nmo * nmo;
  for (int k = threadIdx.x; k < nmo; k += blockDim.x) {
    if (fold && k < l) continue;
    cd acc = cmk(0.0, 0.0);
    for (int i = 0; i < nup; ++i) {
      acc += u0[(long)i * nmo + l] * g0[(long)i * nmo + k];
      if (fold && k > l) acc += u0[(long)i * nmo + k] * g0[(long)i * nmo + l];
    }
    for (int i = 0; i < ndn; ++i) {
      acc += u1[(long)i * nmo + l] * g1[(long)i * nmo + k];
      if (fold && k > l) acc += u1[(long)i * nmo + k] * g1[(long)i * nmo + l];
    }
    const long at = fold ? (long)l * nmo - (long)l * (l - 1) / 2 + (k - l) : (long)l * nmo + k;
    F[(long)w * size + at] = acc * inv;
  }
}

// out[n ld + lk] = Likn[lk][n], the rows l <= k only when folded
__global__ void k_ph_rows_of_vectors(int nmo, int nchol, int fold, int ld,
                                     const double* __restrict__ Likn,
                                     double* __restrict__ out) {
  __shared__ double tile[32][33];
  const int l = blockIdx.z, kb = blockIdx.y * 32, nb = blockIdx.x * 32;
  for (int r = threadIdx.y; r < 32; r += 8) {
    const int k = kb + r, n = nb + threadIdx.x;
    if (k < nmo && n < nchol) tile[r][threadIdx.x] = Likn[((long)l * nmo + k) * nchol + n];
  }
  __syncthreads();
  for (int r = threadIdx.y; r < 32; r += 8) {
    const int n = nb + r, k = kb + threadIdx.x;
    if (n < nchol && k < nmo && !(fold && k < l)) {
      const long at = fold ? (long)l * nmo - (long)l * (l - 1) / 2 + (k - l) : (long)l * nmo + k;
      out[(long)n * ld + at] = tile[threadIdx.x][r];
    }
  }
}

size_t exc_lds(int nv, int nel, int nact) {
  return sizeof(cd) * (size_t)nv * ((size_t)nel * nel + 2 * (size_t)nel * (nact - nel));
}

}  // namespace

// Vectors per workgroup: 4 or 2 while two workgroups fit a CU, else 1; 0: S and B of one vector do
// not fit LDS.
int ph_exc_vectors(int nel, int nact) {
  if (exc_lds(4, nel, nact) <= 78 * 1024) return 4;
  if (exc_lds(2, nel, nact) <= 78 * 1024) return 2;
  return exc_lds(1, nel, nact) <= 150 * 1024 ? 1 : 0;
}

int ph_exc_groups(int nel, int nact, int nchol) {
  const int nv = ph_exc_vectors(nel, nact);
  return nv > 0 ? (nchol + nv) / nv : 0;   // nchol + 1 vectors with the one-body matrix
}

void launch_ph_ratios_q(hipStream_t s, int nw, int nel, int nact, long qtot, int nshell, int maxdet,
                        int maxnex, const PhShell* shells, const double* QQ0, double* ratio,
                        double* Q) {
  if (nw <= 0) return;
  if (nshell == 0) {
    launch_ph_fill(s, nw, 1.0, 0.0, ratio);
    return;
  }
  const long blocks = ((long)nw * std::max(maxdet, 1) + kThreads - 1) / kThreads;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks, nshell), dim3(kThreads), 0, s, nw, nel, nact,
                       qtot, shells, (const cd*)QQ0, (cd*)ratio, (cd*)Q);
  };
  maxnex <= 4 ? go(k_ph_ratios_q<4>) : go(k_ph_ratios_q<8>);
  AFQ_HIP(hipGetLastError());
}

void launch_ph_weights(hipStream_t s, int nw, int nu, const int* cp, const int* ci,
                       const double* cv, const double* own, const double* other, double* wgt,
                       double* sum) {
  if (nw <= 0) return;
  hipLaunchKernelGGL(k_ph_weights, dim3(nu, (nw + 31) / 32), dim3(256), 0, s, nw, cp, ci,
                     (const cd*)cv, (const cd*)own, (const cd*)other, (cd*)wgt);
  AFQ_HIP(hipGetLastError());
  if (sum) {
    hipLaunchKernelGGL(k_ph_weight_sum, dim3(nw), dim3(64), 0, s, nw, nu, (const cd*)wgt, (cd*)sum);
    AFQ_HIP(hipGetLastError());
  }
}

void launch_ph_exc(hipStream_t s, bool down, int nw, int nel, int nact, int nchol, long qtot,
                   int nshell, int maxnex, int nu_own, int nu_up, const PhShell* shells,
                   const double* T, const double* QQ0, const double* Q, const double* wgt,
                   double* KE, const int* cp, const int* ci, const double* cv, const double* rup,
                   const double* rdn, double* part) {
  if (nw <= 0) return;
  const int nv = ph_exc_vectors(nel, nact);
  const size_t lds = exc_lds(nv, nel, nact);
  const dim3 grid(nw, ph_exc_groups(nel, nact, nchol));
  auto go = [&](auto kern) {
    ensure_dynamic_lds((const void*)kern, lds);
    hipLaunchKernelGGL(kern, grid, dim3(kThreads), lds, s, nw, nel, nact, nchol, qtot, nshell,
                       nu_own, nu_up, shells, (const cd*)T, (const cd*)QQ0, (const cd*)Q,
                       (const cd*)wgt, (cd*)KE, cp, ci, (const cd*)cv, (const cd*)rup,
                       (const cd*)rdn, (cd*)part);
  };
  auto pick = [&](auto mx, auto dn) {
    constexpr int MX = decltype(mx)::value;
    constexpr bool DN = decltype(dn)::value;
    if (nv == 4) go(k_ph_exc<MX, 4, DN>);
    else if (nv == 2) go(k_ph_exc<MX, 2, DN>);
    else go(k_ph_exc<MX, 1, DN>);
  };
  const std::integral_constant<int, 4> four;
  const std::integral_constant<int, 8> eight;
  if (down) maxnex <= 4 ? pick(four, std::true_type()) : pick(eight, std::true_type());
  else maxnex <= 4 ? pick(four, std::false_type()) : pick(eight, std::false_type());
  AFQ_HIP(hipGetLastError());
}

void launch_ph_exc_finish(hipStream_t s, int nw, int nu, int gu, int gd, double E0, const double* wgt,
                          const double* pu, const double* pd, const double* log_ov, double* E,
                          double* ov) {
  if (nw <= 0) return;
  hipLaunchKernelGGL(k_ph_exc_finish, dim3(nw), dim3(64), 0, s, nw, nu, gu, gd, cmk(E0, 0.0),
                     (const cd*)wgt, (const cd*)pu, (const cd*)pd, (const cd*)log_ov, (cd*)E,
                     (cd*)ov);
  AFQ_HIP(hipGetLastError());
}

void launch_ph_expansion_R(hipStream_t s, int nw, int nel, int nact, int nu, long qtot,
                           const int* rp, const int* ru, const int* rq, const double* QQ0,
                           const double* Q, const double* wgt, double* R, double* ov) {
  if (nw <= 0) return;
  hipLaunchKernelGGL(k_ph_expansion_R, dim3(nw), dim3(kThreads), 0, s, nw, nel, nact, nu, qtot, rp,
                     ru, rq, (const cd*)QQ0, (const cd*)Q, (const cd*)wgt, (cd*)R, (cd*)ov);
  AFQ_HIP(hipGetLastError());
}

void launch_ph_density(hipStream_t s, int nw, int nup, int ndn, int nact, int nmo, bool fold,
                       const double* R0, const double* A0, const double* G0, const double* R1,
                       const double* A1, const double* G1, const double* ov, double* U0, double* U1,
                       double* F) {
  if (nw <= 0) return;
  hipLaunchKernelGGL(k_ph_ra, dim3((nup * nmo + 255) / 256, nw), dim3(256), 0, s, nup, nact, nmo,
                     (const cd*)R0, (const cd*)A0, (cd*)U0);
  hipLaunchKernelGGL(k_ph_ra, dim3((ndn * nmo + 255) / 256, nw), dim3(256), 0, s, ndn, nact, nmo,
                     (const cd*)R1, (const cd*)A1, (cd*)U1);
  hipLaunchKernelGGL(k_ph_density, dim3(nmo, nw), dim3(nmo <= 64 ? 64 : (nmo <= 128 ? 128 : 256)), 0,
                     s, nup, ndn, nmo, fold ? 1 : 0, (const cd*)U0, (const cd*)G0, (const cd*)U1,
                     (const cd*)G1, (const cd*)ov, (cd*)F);
  AFQ_HIP(hipGetLastError());
}

void launch_ph_rows_of_vectors(hipStream_t s, int nmo, int nchol, bool fold, int ld,
                               const double* Likn, double* out) {
  hipLaunchKernelGGL(k_ph_rows_of_vectors, dim3((nchol + 31) / 32, (nmo + 31) / 32, nmo),
                     dim3(32, 8), 0, s, nmo, nchol, fold ? 1 : 0, ld, Likn, out);
  AFQ_HIP(hipGetLastError());
}

}  // namespace afq
