// Ozaki split of FP64 rows into int8 slices, x = u (q0 + q1/254 + q2/254^2 + ...), and the FP64 value of
// slice sums: shared by the int8 exchange kernels.
#pragma once
#include "afq_internal.hpp"

namespace afq {
namespace i8 {

typedef int i4 __attribute__((ext_vector_type(4)));

constexpr int kS = 6;             // slices of G and of Lnak
constexpr double kBase = 254.0;   // ratio of consecutive slice units

// power-of-two unit of a row whose largest |component| is mx: |x / u| < 127 for every x of the
// row. Rows below 2^-960 count as zero (their products are far below any energy resolution);
// a non-finite row gets NaN so that its energies come out NaN as in FP64.
__device__ inline double row_unit(double mx, bool& zero) {
  zero = false;
  if (!(mx <= 1.0e300)) return __builtin_nan("");
  if (mx < 0x1p-960) {
    zero = true;
    return 1.0;
  }
  int e;
  frexp(mx * (128.0 / 127.0), &e);
  return ldexp(1.0, e - 7);
}

// the slices of r = x / u (|r| < 127; x * inv_u is exact, inv_u being a power of two)
__device__ inline void slice(double r, int (&q)[kS]) {
#pragma unroll
  for (int s = 0; s < kS; ++s) {
    const double qs = rint(r);
    q[s] = (int)qs;
    r = (r - qs) * kBase;
  }
}

__device__ inline unsigned pack4(int a, int b, int c, int d) {
  return (unsigned)(a & 0xff) | ((unsigned)(b & 0xff) << 8) | ((unsigned)(c & 0xff) << 16) |
         ((unsigned)(d & 0xff) << 24);
}

__device__ inline i4 mfma_i8(i4 a, i4 b, i4 c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

// workgroup barrier after this wavefront's LDS reads and writes; its global loads and stores in flight
// are not waited for. The memory clobber keeps the compiler from moving memory accesses across.
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A fragments of a row of G: lane group g holds k = 64 kc + 16 g + j (j < 16) of the row at Gr (ok: there
// is one); returns the row's unit
template <int KC>
__device__ inline double slice_row(const double2* Gr, bool ok, int M, int g, i4 (&ar)[KC][kS], i4 (&ai)[KC][kS]) {
  double mx = 0.0;
  if (ok) {
    for (int kc = 0; kc < KC; ++kc)
      for (int j = 0; j < 16; ++j) {
        const int k = 64 * kc + 16 * g + j;
        if (k < M) {
          const double2 x = Gr[k];
          const double xr = fabs(x.x), xi = fabs(x.y);
          // a NaN or Inf anywhere in the row must survive the max (fmax drops NaN)
          mx = (xr <= 1.0e300 && xi <= 1.0e300) ? fmax(mx, fmax(xr, xi)) : INFINITY;
        }
      }
  }
  mx = fmax(mx, __shfl_xor(mx, 16, 64));
  mx = fmax(mx, __shfl_xor(mx, 32, 64));
  bool zero;
  const double u = row_unit(mx, zero);
  const bool finite = u == u;
  const double inv = (finite && !zero) ? 1.0 / u : 0.0;
#pragma unroll
  for (int kc = 0; kc < KC; ++kc) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {   // bytes 4d..4d+3 of each fragment
      int qr[4][kS], qi[4][kS];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = 64 * kc + 16 * g + 4 * d + j;
        double2 x = double2{0.0, 0.0};
        if (ok && k < M && inv != 0.0) x = Gr[k];
        slice(x.x * inv, qr[j]);
        slice(x.y * inv, qi[j]);
      }
#pragma unroll
      for (int s = 0; s < kS; ++s) {
        ar[kc][s][d] = (int)pack4(qr[0][s], qr[1][s], qr[2][s], qr[3][s]);
        ai[kc][s][d] = (int)pack4(qi[0][s], qi[1][s], qi[2][s], qi[3][s]);
      }
      __builtin_amdgcn_sched_barrier(0);   // four elements at a time (registers)
    }
  }
  return u;
}

// 254 sum_o 254^-o c_o over the orders o <= ON of KC 64-wide chunks (LC: complex Lnak, real and imaginary
// products in one sum). |c_o| <= (o + 1) 64 KC 127^2 (2 with LC): 254 c0 + c1 fits int32 always, 254 c2 +
// c3 with real Lnak or one chunk, 254 c4 + c5 with both (24-bit factors: |c0|, |c2|, |c4| < 2^23)
template <int ON, int KC, bool LC>
__device__ inline double join_orders(const i4* c, int r) {
  constexpr int C3 = ON >= 3 ? 3 : 0, C4 = ON >= 4 ? 4 : 0, C5 = ON >= 5 ? 5 : 0;
  double lo = 0.0;
  if (ON >= 5 && KC == 1 && !LC) lo = (double)(__mul24(254, c[C4][r]) + c[C5][r]) * (1.0 / kBase);
  else if (ON >= 5) lo = fma((double)c[C5][r], 1.0 / kBase, (double)c[C4][r]);
  else if (ON == 4) lo = (double)c[C4][r];
  double mid;
  if ((LC && KC > 1) || ON < 3) {
    mid = (double)c[2][r];
    if (ON >= 3) mid = fma((double)c[C3][r], 1.0 / kBase, mid);
    mid *= kBase;
  } else {
    mid = (double)(__mul24(254, c[2][r]) + c[C3][r]);
  }
  if (ON >= 4) mid = fma(lo, 1.0 / kBase, mid);
  return fma(mid, 1.0 / (kBase * kBase), (double)(__mul24(254, c[0][r]) + c[1][r]));
}

}  // namespace i8
}  // namespace afq
