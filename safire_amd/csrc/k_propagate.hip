// Walker propagation Phi <- P1 exp(iV) P1 Phi with exp(iV) as its order-n Taylor series
// (det_ops::detail::propagate_impl + apply_expM, propagate.hpp:41-70, 241-298):
//   S = P1 Phi;  T = S;  for k = 1..order: T = (i/k) V_w T;  S += T;   Phi = P1 S
//
// One workgroup per walker, a wavefront per 16-row tile of the walker (or RPW of them) with all of its
// column tiles (two column tiles of a walker of up to 32 rows: one each), so a fragment of V_w or P1 is
// loaded by one wavefront and used for every column tile. The current Taylor term T lives in LDS as the
// MFMA B operand ([k][column], columns padded to 16); the running sum S stays in registers in the
// accumulator layout. In k step t lane group g holds k = 4 t + g, so a product takes ceil(M / 4) steps.
//
// V_w is complex symmetric when the Cholesky vectors are (real orbitals): then only its upper
// triangle exists, packed (row i <= j at i (2 M - i - 1) / 2 + j), half the memory and half of the
// work that forms it. For M <= 64 V_w is expanded into LDS once per walker, its loads, those of Phi and
// the first ones of P1 in flight together; above that its fragments are read from memory (L2) one
// group of four k steps ahead, every element at its (min, max) place. CONJ applies -conj(V) = -V^H
// instead (the adjoint series of back-propagation). A real P1 (P1r) takes 2 FP64 MFMAs per tile and k
// step, complex products take 4.
//
// Bound: FP64 MFMA, 64 cycles each (M 128, N 32: 2 x 1024 + 6 x 2048 per walker); for M <= 32 the
// latency of 8 dependent products. Packed V_w and a real P1, against four wavefronts with one 16 x 16
// tile at a time, full V_w and a complex P1: M 128, N 32, 1024 walkers 797 -> 554 us; M 77, N 24, 1024
// walkers 341 -> 300 us; M 64, N 16, 512 walkers 59 -> 50 us; M 32, N 20, 1024 walkers 54 -> 46 us;
// M 19, N 3, 64 walkers 18.0 -> 13.5 us. Full V_w and a complex P1 (det_ops level): M 96, N 32, 1024
// walkers 439 -> 424 us; M 32, N 20, 1024 walkers 48 -> 45 us; M 16, N 4, 256 walkers 10.4 -> 10.9 us;
// M 77, N 40 (three column tiles of five row tiles: five wavefronts on four SIMDs) 448 -> 540 us.
#include "afq_internal.hpp"

#include <algorithm>

namespace afq {

namespace {

// the upper triangle's row i starts here, so that element (i, j) sits at packed_row + j
__host__ __device__ inline int packed_row(int i, int M) { return i * (2 * M - i - 1) / 2; }

// V_w in LDS: element (k, row) of its transpose. The column is XORed with the row's low bits, so that
// 16 lanes writing down a column hit 16 different banks, as 16 lanes reading along a row do.
__device__ inline int vpos(int k, int row, int MB) { return k * MB + (row ^ (k & 15)); }

// RPW row tiles and CT column tiles per wavefront, CS groups of column tiles, VLDS: V_w in LDS (RPW is
// 1), SYM: packed V, CONJ: -conj(V)
template <int RPW, int CT, int CS, bool VLDS, bool SYM, bool CONJ>
__global__ __launch_bounds__(512, !VLDS && RPW * CT <= 2 && RPW == 1 ? 4 : 2) void k_propagate(
    int M, int N, cd* __restrict__ Phi, long ldw, const cd* __restrict__ P1,
    const double* __restrict__ P1r, const cd* __restrict__ V, int order, int ks) {
  // [MK][16 CT CS] current term, (VLDS) [MK][MB] V_w transposed, [ks - 1][row tiles][CT][4][64] partials
  extern __shared__ cd smem[];
  const int w = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int allw = blockDim.x >> 6, nwc = allw / ks;
  const int nwave = nwc / CS;                 // wavefronts that share the row tiles
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kh = wid / nwc, wc = wid - kh * nwc;                       // part of k
  const int ch = CS == 1 ? 0 : wc / nwave, wave = wc - ch * nwave;     // part of the columns, first row tile
  const int g = lane >> 4, r16 = lane & 15;
  const int MB = (M + 15) & ~15;
  const int steps = (M + 3) >> 2;             // k steps of a product
  const int MK = 16 * ((steps + 3) >> 2);     // rows of T in LDS (zero past M)
  const int per = (steps + ks - 1) / ks;      // k steps of this wavefront: t0 .. t0 + mine - 1
  const int t0 = kh * per, mine = min(per, steps - t0);
  constexpr int NB = 16 * CT * CS;
  const int C0 = 16 * CT * ch;
  cd* sB = smem;
  cd* sV = smem + MK * NB;
  cd* sP = sV + (VLDS ? MK * MB : 0);
  cd* P = Phi + (long)w * ldw;
  const cd* Vw = V + (long)w * (SYM ? (long)M * (M + 1) / 2 : (long)M * M);

  auto p1_real = [&](int row, int t) {
    const int k = 4 * t + g;
    return cmk(row < M && k < M ? P1r[row * M + k] : 0.0, 0.0);
  };
  auto p1_cplx = [&](int row, int t) {
    const int k = 4 * t + g;
    return row < M && k < M ? P1[row * M + k] : cmk(0.0, 0.0);
  };
  cd first[4];
  if (VLDS) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
      first[s] = P1r != nullptr ? p1_real(16 * wave + r16, t0 + s) : p1_cplx(16 * wave + r16, t0 + s);
  }
  // Phi: the first four entries of a thread are in flight while V_w is staged
  auto phi = [&](int e) {
    const int i = e / NB, b = e - i * NB;
    return e < MK * NB && i < M && b < N ? P[i * N + b] : cmk(0.0, 0.0);
  };
  cd ph[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) ph[s] = phi(tid + s * (int)blockDim.x);
  if (VLDS) {
    // sV(k, row) = V[row][k], zero outside M x M; 16 lanes along a row of V, at most 64 long
    for (int i0 = 4 * wid + g; i0 < MB; i0 += 8 * allw) {
      cd x[2][4];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int i = i0 + 4 * allw * h, j = 16 * q + r16;
          x[h][q] = cmk(0.0, 0.0);
          if (i < M && j < M && !(SYM && j < i)) x[h][q] = Vw[SYM ? packed_row(i, M) + j : i * M + j];
        }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int i = i0 + 4 * allw * h, j = 16 * q + r16;
          if (i >= MB || j >= MB || (SYM && j < i)) continue;   // the mirror of (j, i)
          if (CONJ) x[h][q].re = -x[h][q].re;
          sV[vpos(j, i, MB)] = x[h][q];
          if (SYM) sV[vpos(i, j, MB)] = x[h][q];
        }
    }
  }
#pragma unroll
  for (int s = 0; s < 4; ++s)
    if (tid + s * (int)blockDim.x < MK * NB) sB[tid + s * (int)blockDim.x] = ph[s];
  for (int e = tid + 4 * blockDim.x; e < MK * NB; e += blockDim.x) sB[e] = phi(e);
  __syncthreads();

  d4 sr[RPW][CT], si[RPW][CT], tr[RPW][CT], ti[RPW][CT];

  // t += A T of one k step: a = A[row][4 t + g], bq = the step's row g of T
  auto step = [&](auto real_c, int q, const cd& a, const cd (&b)[CT]) {
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      tr[q][c] = mfma16x16x4(a.re, b[c].re, tr[q][c]);
      ti[q][c] = mfma16x16x4(a.re, b[c].im, ti[q][c]);
    }
    if (!decltype(real_c)::value)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        tr[q][c] = mfma16x16x4(-a.im, b[c].im, tr[q][c]);
        ti[q][c] = mfma16x16x4(a.im, b[c].re, ti[q][c]);
      }
  };
  auto clear = [&](int q) {
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      tr[q][c] = d4{0, 0, 0, 0};
      ti[q][c] = d4{0, 0, 0, 0};
    }
  };
  // t = A T over the wavefront's row tiles and its part of k, A in memory: load(row, t) gives
  // A[row][4 t + g] (0 past M), four steps ahead of the products
  auto product = [&](auto real_c, bool have, auto&& load) {
#pragma unroll
    for (int q = 0; q < RPW; ++q) {
      clear(q);
      const int row = 16 * (wave + q * nwave) + r16;
      if (16 * (wave + q * nwave) < M) {   // uniform
        const cd* bp = sB + (4 * t0 + g) * NB + C0 + r16;
        const int full = mine >> 2;
        auto one = [&](int s, const cd& a) {
          cd b[CT];
#pragma unroll
          for (int c = 0; c < CT; ++c) b[c] = bp[4 * s * NB + 16 * c];
          step(real_c, q, a, b);
        };
        cd a[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) a[s] = have ? first[s] : load(row, t0 + s);
        // one row tile per wavefront: every step guarded and no operands loaded past the last group
        // (M 77, N 24, 512 walkers 152 us, 159 without; five column tiles spill 19 VGPRs, 127 without)
        constexpr bool GUARD = !VLDS && RPW == 1;
        const int groups = GUARD ? (mine + 3) >> 2 : full;
        for (int t = 0; t < groups; ++t) {
          cd nx[4];
          if (!GUARD || t + 1 < groups)
#pragma unroll
            for (int s = 0; s < 4; ++s) nx[s] = load(row, t0 + 4 * (t + 1) + s);
          else
#pragma unroll
            for (int s = 0; s < 4; ++s) nx[s] = cmk(0.0, 0.0);
#pragma unroll
          for (int s = 0; s < 4; ++s)
            if (!GUARD || 4 * t + s < mine) one(s, a[s]);   // uniform
          bp += 16 * NB;
#pragma unroll
          for (int s = 0; s < 4; ++s) a[s] = nx[s];
        }
        if (!GUARD)
#pragma unroll
          for (int s = 0; s < 3; ++s)
            if (4 * full + s < mine) one(s, a[s]);   // uniform
      }
    }
  };
  // the same with A = V_w in LDS
  auto product_lds = [&]() {
    clear(0);
    const int row = 16 * wave + r16;
    const cd* bp = sB + (4 * t0 + g) * NB + C0 + r16;
    const cd* ap = sV + (4 * t0 + g) * MB;
    int col[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) col[s] = 4 * s * MB + (row ^ ((4 * (t0 + s) + g) & 15));
    const int full = mine >> 2;
    for (int t = 0; t < full; ++t) {
      cd a[4], b[4][CT];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        a[s] = ap[col[s]];
#pragma unroll
        for (int c = 0; c < CT; ++c) b[s][c] = bp[4 * s * NB + 16 * c];
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) step(std::false_type(), 0, a[s], b[s]);
      ap += 16 * MB;
      bp += 16 * NB;
    }
    const int rem = mine - 4 * full;
    if (rem > 0) {   // uniform, as the following
      cd a[3], b[3][CT];
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        const int sc = min(s, rem - 1);
        a[s] = ap[4 * sc * MB + (row ^ ((4 * (t0 + sc) + g) & 15))];
#pragma unroll
        for (int c = 0; c < CT; ++c) b[s][c] = bp[4 * sc * NB + 16 * c];
      }
#pragma unroll
      for (int s = 0; s < 3; ++s)
        if (s < rem) step(std::false_type(), 0, a[s], b[s]);
    }
  };
  // the parts of k meet in the wavefronts of part 0, in order, between two barriers
  auto join = [&]() {
    if (ks == 1) {
      __syncthreads();
      return;
    }
    cd* part = sP + (long)wc * CT * 256 + lane;
    const int stride = nwc * CT * 256;
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
    if (P1r != nullptr) product(std::true_type(), VLDS, p1_real);
    else product(std::false_type(), VLDS, p1_cplx);
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
          if (i < MK) sB[i * NB + C0 + 16 * c + r16] = cmk(xr[q][c][r], xi[q][c][r]);
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
      product_lds();
    else
      product(std::false_type(), false, [&](int row, int t) {
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
      const int b = C0 + 16 * c + r16;
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
  // V_w in LDS. Two column tiles: a wavefront each while that makes four (M 32, N 20, 1024 walkers: 45 us,
  // 45 with one, 54 with two parts of k, 94 with four; 64 walkers: 18, 26, 20 and 25). One column tile:
  // two parts of k, always for 2 row tiles (M 24, N 6, 64 walkers: 13.0 and 14.7 us), else where one
  // workgroup per CU is all there is (M 64, N 8, 64 walkers: 28 and 29 us; 1024 walkers: 115 and 91).
  int cs = 1, ks = 1;
  if (vlds) {
    if (ct == 2 && rt <= 2) cs = 2;
    else if (ct == 1 && (rt == 2 || (M > 12 && nb <= device_cus()))) ks = 2;
    lds += sizeof(cd) * (size_t)(ks - 1) * rt * ct * 256;
  }
  AFQ_CHECK(lds <= 160 * 1024, AFQ_EUNSUPPORTED, "propagate: walker matrix larger than 128 x 64");
  int rpw = (rt + 7) / 8;
  // Five or six wavefronts with a row tile each leave a third of a CU's wavefront slots empty and load its
  // SIMDs unevenly: with more walkers per CU than two or three of them hold, fewer wavefronts with more
  // rows. M 96, N 16: 768 walkers 210 -> 185 us, 1024 317 -> 217; M 77, N 24: 1024 384 -> 300. Five row
  // tiles and 5 walkers per CU keep one row each (M 77, N 24, 1280 walkers: 400 us, 468 with more).
  const int held = (nb + device_cus() - 1) / device_cus();
  if (!vlds && (rt == 5 || rt == 6) && !(rt == 5 && held == 5)) {
    if (ct == 2 && held >= 4) rpw = 3, cs = 2;
    else if (ct == 1 && held == 4) rpw = 3;
    else if (ct == 1 && (held > 4 || (held == 3 && (rt == 6 || kind == VKind::full)))) rpw = 2;
  }
  const int nwave = (rt + rpw - 1) / rpw;
  auto go = [&](auto kern) {
    ensure_dynamic_lds((const void*)kern, lds);
    hipLaunchKernelGGL(kern, dim3(nb), dim3(64 * nwave * ks * cs), lds, s, M, N, reinterpret_cast<cd*>(Phi),
                       ldw, reinterpret_cast<const cd*>(P1), P1r, reinterpret_cast<const cd*>(V),
                       order, ks);
  };
  auto kinds = [&](auto rp, auto c, auto csv, auto vl) {
    constexpr int RP = decltype(rp)::value, CT = decltype(c)::value, CS = decltype(csv)::value;
    constexpr bool VL = decltype(vl)::value;
    switch (kind) {
      case VKind::full: go(k_propagate<RP, CT, CS, VL, false, false>); break;
      case VKind::packed: go(k_propagate<RP, CT, CS, VL, true, false>); break;
      default: go(k_propagate<RP, CT, CS, VL, true, true>); break;
    }
  };
  const std::integral_constant<int, 1> c1;
  const std::integral_constant<int, 2> c2;
  const std::integral_constant<int, 3> c3;
  const std::integral_constant<int, 4> c4;
  const std::integral_constant<int, 5> c5;   // 5 x 5 and 6 x 5 tiles (N <= M)
  if (vlds) {   // M <= 64, four row tiles with one column tile at most
    if (ct == 1) kinds(c1, c1, c1, std::true_type());
    else if (ct == 2 && cs == 2) kinds(c1, c1, c2, std::true_type());
    else if (ct == 2) kinds(c1, c2, c1, std::true_type());
    else kinds(c1, c3, c1, std::true_type());
  } else if (rpw == 1) {
    if (ct == 1) kinds(c1, c1, c1, std::false_type());
    else if (ct == 2) kinds(c1, c2, c1, std::false_type());
    else if (ct == 3) kinds(c1, c3, c1, std::false_type());
    else if (ct == 4) kinds(c1, c4, c1, std::false_type());
    else kinds(c1, c5, c1, std::false_type());
  } else if (rpw == 3 && rt <= 6) {
    if (cs == 2) kinds(c3, c1, c2, std::false_type());
    else kinds(c3, c1, c1, std::false_type());
  } else if (rpw == 2) {
    if (ct == 1) kinds(c2, c1, c1, std::false_type());
    else if (ct == 2) kinds(c2, c2, c1, std::false_type());
    else kinds(c2, c3, c1, std::false_type());
  } else {
    kinds(c4, c1, c1, std::false_type());
  }
  AFQ_HIP(hipGetLastError());
}

}  // namespace afq
