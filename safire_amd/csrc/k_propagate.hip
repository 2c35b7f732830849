// Walker propagation Phi <- P1 exp(iV) P1 Phi with exp(iV) as its order-n Taylor series
// (det_ops::detail::propagate_impl + apply_expM, propagate.hpp:41-70, 241-298):
//   S = P1 Phi;  T = S;  for k = 1..order: T = (i/k) V_w T;  S += T;   Phi = P1 S
//
// One workgroup per walker, a wavefront per 16-row tile of the walker (two where it has more than 8)
// with all of its column tiles, so a fragment of V_w or P1 is loaded by one wavefront only and used
// for every column tile. The current Taylor term T lives in LDS as the MFMA B operand ([k][column],
// columns padded to 16); the running sum S stays in registers in the accumulator layout. In k step t
// lane group g holds k = 4 t + g, so a product takes ceil(M / 4) steps.
//
// V_w is complex symmetric when the Cholesky vectors are (real orbitals): then only its upper
// triangle exists, packed (row i <= j at i (2 M - i - 1) / 2 + j), half the memory and half of the
// work that forms it. For M <= 64 V_w is expanded into LDS once per walker; above that its
// fragments are read from memory (L2) one group of four k steps ahead, every element at its
// (min, max) place. CONJ applies -conj(V) = -V^H instead (the adjoint series of back-propagation).
// A real P1 (P1r) takes 2 FP64 MFMAs per tile and k step, complex products take 4.
//
// Small walkers split k: up to 4 wavefronts share a row tile's products and meet in LDS, in order.
//
// Bound: FP64 MFMA, 64 cycles each (M 128, N 32: 2 x 1024 + 6 x 2048 per walker). Per launch, against
// full V_w and P1 complex: M 128, N 32, 1024 walkers 785 -> 528 us; M 77, N 19, 201 walkers 113 ->
// 96 us; M 64, N 16, 512 walkers 58 -> 56 us; M 19, N 3, 50 walkers 15.8 -> 14.9 us.
#include "afq_internal.hpp"

#include <algorithm>

namespace afq {

namespace {

// the upper triangle's row i starts here, so that element (i, j) sits at packed_row + j
__host__ __device__ inline int packed_row(int i, int M) { return i * (2 * M - i - 1) / 2; }

// V_w in LDS: element (k, row) of its transpose. The column is XORed with the row's low bits, so that
// 16 lanes writing down a column hit 16 different banks, as 16 lanes reading along a row do.
__device__ inline int vpos(int k, int row, int MB) { return k * MB + (row ^ (k & 15)); }

// RPW row tiles per wavefront, CT column tiles, VLDS: V_w in LDS, SYM: packed V, CONJ: -conj(V)
template <int RPW, int CT, bool VLDS, bool SYM, bool CONJ>
__global__ __launch_bounds__(512, !VLDS && RPW * CT <= 2 && RPW == 1 ? 4 : 2) void k_propagate(
    int M, int N, cd* __restrict__ Phi, long ldw, const cd* __restrict__ P1,
    const double* __restrict__ P1r, const cd* __restrict__ V, int order, int ks) {
  // [MK][16 CT] current term, (VLDS) [MK][MB] V_w transposed, [ks - 1][row tiles][CT][4][64] partials
  extern __shared__ cd smem[];
  const int w = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int allw = blockDim.x >> 6, nwave = allw / ks;   // nwave wavefronts share the row tiles
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kh = wid / nwave, wave = wid - kh * nwave;   // part of k, first row tile
  const int g = lane >> 4, r16 = lane & 15;
  const int MB = (M + 15) & ~15;
  const int steps = (M + 3) >> 2;             // k steps of a product
  const int MK = 16 * ((steps + 3) >> 2);     // rows of T in LDS (zero past M)
  const int per = (steps + ks - 1) / ks;      // k steps of this wavefront: t0 .. t0 + mine - 1
  const int t0 = kh * per, mine = min(per, steps - t0);
  const int groups = (mine + 3) >> 2;         // in groups of four
  constexpr int NB = 16 * CT;
  cd* sB = smem;
  cd* sV = smem + MK * NB;
  cd* sP = sV + (VLDS ? MK * MB : 0);
  cd* P = Phi + (long)w * ldw;
  const cd* Vw = V + (long)w * (SYM ? (long)M * (M + 1) / 2 : (long)M * M);

  for (int e = tid; e < MK * NB; e += blockDim.x) {
    const int i = e / NB, b = e - i * NB;
    sB[e] = (i < M && b < N) ? P[i * N + b] : cmk(0.0, 0.0);
  }
  if (VLDS) {
    // sV(k, row) = V[row][k], zero outside M x M; a wavefront per row of V
    for (int i = wid; i < MB; i += allw)
      for (int j = lane; j < MB; j += 64) {
        if (SYM && j < i) continue;   // the mirror of (j, i)
        cd x = cmk(0.0, 0.0);
        if (i < M && j < M) x = Vw[SYM ? packed_row(i, M) + j : i * M + j];
        if (CONJ) x.re = -x.re;
        if (j < MK) sV[vpos(j, i, MB)] = x;
        if (SYM && i < MK) sV[vpos(i, j, MB)] = x;
      }
  }
  __syncthreads();

  d4 sr[RPW][CT], si[RPW][CT], tr[RPW][CT], ti[RPW][CT];

  // t = A T over the wavefront's row tiles and its part of k; load(row, t) gives A[row][4 t + g] (0
  // past M)
  auto product = [&](auto real_c, auto&& load) {
    constexpr bool REAL = decltype(real_c)::value;
#pragma unroll
    for (int q = 0; q < RPW; ++q) {
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        tr[q][c] = d4{0, 0, 0, 0};
        ti[q][c] = d4{0, 0, 0, 0};
      }
      const int row = 16 * (wave + q * nwave) + r16;
      if (16 * (wave + q * nwave) < M) {   // uniform
        cd a[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) a[s] = load(row, t0 + s);
        const cd* bp = sB + (4 * t0 + g) * NB + r16;
        for (int t = 0; t < groups; ++t) {
          cd nx[4];
          if (t + 1 < groups)
#pragma unroll
            for (int s = 0; s < 4; ++s) nx[s] = load(row, t0 + 4 * (t + 1) + s);
          else
#pragma unroll
            for (int s = 0; s < 4; ++s) nx[s] = cmk(0.0, 0.0);
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            if (4 * t + s < mine) {   // uniform
              cd b[CT];
#pragma unroll
              for (int c = 0; c < CT; ++c) b[c] = bp[(4 * (4 * t + s)) * NB + 16 * c];
#pragma unroll
              for (int c = 0; c < CT; ++c) {
                tr[q][c] = mfma16x16x4(a[s].re, b[c].re, tr[q][c]);
                ti[q][c] = mfma16x16x4(a[s].re, b[c].im, ti[q][c]);
              }
              if (!REAL)
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                  tr[q][c] = mfma16x16x4(-a[s].im, b[c].im, tr[q][c]);
                  ti[q][c] = mfma16x16x4(a[s].im, b[c].re, ti[q][c]);
                }
            }
          }
#pragma unroll
          for (int s = 0; s < 4; ++s) a[s] = nx[s];
        }
      }
    }
  };
  // the parts of k meet in the wavefronts of part 0, in order, between two barriers
  auto join = [&]() {
    if (ks == 1) {
      __syncthreads();
      return;
    }
    cd* part = sP + (long)wave * CT * 256 + lane;
    const int stride = nwave * CT * 256;
    if (kh > 0)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          part[(kh - 1) * stride + (4 * c + r) * 64] = cmk(tr[0][c][r], ti[0][c][r]);
    __syncthreads();
    if (kh == 0)
      for (int h = 0; h < ks - 1; ++h)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const cd x = part[h * stride + (4 * c + r) * 64];
            tr[0][c][r] += x.re;
            ti[0][c][r] += x.im;
          }
  };
  auto one_body = [&]() {
    if (P1r != nullptr)
      product(std::true_type(), [&](int row, int t) {
        const int k = 4 * t + g;
        return cmk(row < M && k < M ? P1r[row * M + k] : 0.0, 0.0);
      });
    else
      product(std::false_type(), [&](int row, int t) {
        const int k = 4 * t + g;
        return row < M && k < M ? P1[row * M + k] : cmk(0.0, 0.0);
      });
  };
  auto store = [&](const d4 (&xr)[RPW][CT], const d4 (&xi)[RPW][CT]) {
    if (kh > 0) return;
#pragma unroll
    for (int q = 0; q < RPW; ++q)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * (wave + q * nwave) + acc_row<double>(g, r);
          if (i < MK) sB[i * NB + 16 * c + r16] = cmk(xr[q][c][r], xi[q][c][r]);
        }
  };

  // S = P1 Phi
  one_body();
  join();
  store(tr, ti);
#pragma unroll
  for (int q = 0; q < RPW; ++q)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      sr[q][c] = tr[q][c];
      si[q][c] = ti[q][c];
    }
  __syncthreads();
  for (int k = 1; k <= order; ++k) {
    if (VLDS)
      product(std::false_type(), [&](int row, int t) { return sV[vpos(4 * t + g, row, MB)]; });
    else
      product(std::false_type(), [&](int row, int t) {
        const int kk = 4 * t + g;
        cd x = cmk(0.0, 0.0);
        if (row < M && kk < M)
          x = Vw[SYM ? packed_row(min(row, kk), M) + max(row, kk) : row * M + kk];
        if (CONJ) x.re = -x.re;
        return x;
      });
    join();
    const double f = 1.0 / (double)k;
    // T <- (i/k) (V T):  re = -f im, im = f re
#pragma unroll
    for (int q = 0; q < RPW; ++q)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const d4 nr = -f * ti[q][c], ni = f * tr[q][c];
        tr[q][c] = nr;
        ti[q][c] = ni;
        sr[q][c] += nr;
        si[q][c] += ni;
      }
    if (k < order) store(tr, ti);
    else store(sr, si);
    __syncthreads();
  }
  // Phi = P1 S
  one_body();
  if (ks > 1) join();
  if (kh > 0) return;
#pragma unroll
  for (int q = 0; q < RPW; ++q)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int b = 16 * c + r16;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * (wave + q * nwave) + acc_row<double>(g, r);
        if (i < M && b < N) P[i * N + b] = cmk(tr[q][c][r], ti[q][c][r]);
      }
    }
}

}  // namespace

void launch_propagate(hipStream_t s, int nb, int M, int N, double* Phi, long ldw,
                      const double* P1, const double* P1r, const double* V, VKind kind, int order) {
  if (nb <= 0 || N <= 0) return;
  const int MB = (M + 15) & ~15, NB = (N + 15) & ~15;
  const int rt = MB / 16, ct = NB / 16;
  AFQ_CHECK((rt * ct + 3) / 4 <= 8, AFQ_EUNSUPPORTED, "propagate: walker matrix larger than 128 x 64");
  const int MK = ((M + 3) / 4 + 3) / 4 * 16;
  const size_t lds_b = sizeof(cd) * (size_t)MK * NB, lds_v = sizeof(cd) * (size_t)MK * MB;
  // V_w in LDS when both fit in 80 KB (two workgroups per CU)
  const bool vlds = lds_b + lds_v <= 80 * 1024 && rt <= 8;
  size_t lds = vlds ? lds_b + lds_v : lds_b;
  // small walkers leave wavefronts free: up to 4 of them split the k range of a row tile, as long as
  // two workgroups still fit a CU, or one per CU is all there are
  int ks = 1;
  if (vlds)
    for (int q = 4; q > 1; q /= 2) {
      const size_t more = sizeof(cd) * (size_t)(q - 1) * rt * ct * 256;
      if (rt * q <= 8 && (M + 3) / 4 >= q &&
          (lds + more <= 80 * 1024 || (nb <= device_cus() && lds + more <= 150 * 1024))) {
        ks = q;
        lds += more;
        break;
      }
    }
  AFQ_CHECK(lds <= 160 * 1024, AFQ_EUNSUPPORTED, "propagate: walker matrix larger than 128 x 64");
  const int rpw = (rt + 7) / 8;
  const int nwave = (rt + rpw - 1) / rpw;
  auto go = [&](auto kern) {
    ensure_dynamic_lds((const void*)kern, lds);
    hipLaunchKernelGGL(kern, dim3(nb), dim3(64 * nwave * ks), lds, s, M, N, reinterpret_cast<cd*>(Phi),
                       ldw, reinterpret_cast<const cd*>(P1), P1r, reinterpret_cast<const cd*>(V),
                       order, ks);
  };
  auto kinds = [&](auto rp, auto c, auto vl) {
    constexpr int RP = decltype(rp)::value, CT = decltype(c)::value;
    constexpr bool VL = decltype(vl)::value;
    switch (kind) {
      case VKind::full: go(k_propagate<RP, CT, VL, false, false>); break;
      case VKind::packed: go(k_propagate<RP, CT, VL, true, false>); break;
      default: go(k_propagate<RP, CT, VL, true, true>); break;
    }
  };
  const std::integral_constant<int, 1> c1;
  const std::integral_constant<int, 2> c2;
  const std::integral_constant<int, 3> c3;
  const std::integral_constant<int, 4> c4;
  const std::integral_constant<int, 5> c5;   // 5 x 5 and 6 x 5 tiles (N <= M)
  if (vlds) {
    if (ct == 1) kinds(c1, c1, std::true_type());
    else if (ct == 2) kinds(c1, c2, std::true_type());
    else if (ct == 3) kinds(c1, c3, std::true_type());
    else kinds(c1, c4, std::true_type());
  } else if (rpw == 1) {
    if (ct == 1) kinds(c1, c1, std::false_type());
    else if (ct == 2) kinds(c1, c2, std::false_type());
    else if (ct == 3) kinds(c1, c3, std::false_type());
    else if (ct == 4) kinds(c1, c4, std::false_type());
    else kinds(c1, c5, std::false_type());
  } else if (rpw == 2) {
    if (ct == 1) kinds(c2, c1, std::false_type());
    else if (ct == 2) kinds(c2, c2, std::false_type());
    else kinds(c2, c3, std::false_type());
  } else {
    kinds(c4, c1, std::false_type());
  }
  AFQ_HIP(hipGetLastError());
}

}  // namespace afq
