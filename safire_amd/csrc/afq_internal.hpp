// Internal declarations of the MI355X walker-step library: device complex helpers, the MFMA
// wrappers, the per-system engine state and the kernel launchers.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <string>
#include <vector>

#include "../../include/afq.h"

namespace afq {

// ------------------------------------------------------------------ error plumbing
void set_error(const std::string& msg);
struct Error {
  int code;
  std::string msg;
};

#define AFQ_HIP(call)                                                                       \
  do {                                                                                      \
    hipError_t e_ = (call);                                                                 \
    if (e_ != hipSuccess)                                                                   \
      throw ::afq::Error{AFQ_EHIP, std::string(#call) + ": " + hipGetErrorString(e_)};      \
  } while (0)

#define AFQ_CHECK(cond, code, msg)                                                          \
  do {                                                                                      \
    if (!(cond)) throw ::afq::Error{(code), (msg)};                                         \
  } while (0)

// ------------------------------------------------------------------ complex on the device
struct cd {
  double re, im;
};

__host__ __device__ inline cd cmk(double r, double i) { return cd{r, i}; }
__host__ __device__ inline cd operator+(cd a, cd b) { return cd{a.re + b.re, a.im + b.im}; }
__host__ __device__ inline cd operator-(cd a, cd b) { return cd{a.re - b.re, a.im - b.im}; }
__host__ __device__ inline cd operator-(cd a) { return cd{-a.re, -a.im}; }
__host__ __device__ inline cd operator*(cd a, cd b) {
  return cd{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__host__ __device__ inline cd operator*(double s, cd a) { return cd{s * a.re, s * a.im}; }
__host__ __device__ inline cd& operator+=(cd& a, cd b) {
  a.re += b.re;
  a.im += b.im;
  return a;
}
__host__ __device__ inline cd& operator-=(cd& a, cd b) {
  a.re -= b.re;
  a.im -= b.im;
  return a;
}
__host__ __device__ inline cd cconj(cd a) { return cd{a.re, -a.im}; }
__host__ __device__ inline double cnorm(cd a) { return a.re * a.re + a.im * a.im; }
__host__ __device__ inline double cabs_(cd a) { return hypot(a.re, a.im); }
__host__ __device__ inline double cabs1(cd a) { return fabs(a.re) + fabs(a.im); }
__host__ __device__ inline bool cis0(cd a) { return a.re == 0.0 && a.im == 0.0; }
// complex division with Smith's scaling (the -fcx-fortran-rules division of the host build)
__host__ __device__ inline cd cdiv(cd a, cd b) {
  if (fabs(b.re) >= fabs(b.im)) {
    double r = b.im / b.re, d = b.re + b.im * r;
    return cd{(a.re + a.im * r) / d, (a.im - a.re * r) / d};
  } else {
    double r = b.re / b.im, d = b.im + b.re * r;
    return cd{(a.re * r + a.im) / d, (a.im * r - a.re) / d};
  }
}
__host__ __device__ inline cd clog_(cd a) { return cd{log(hypot(a.re, a.im)), atan2(a.im, a.re)}; }
__host__ __device__ inline cd cexp_(cd a) {
  double e = exp(a.re);
  return cd{e * cos(a.im), e * sin(a.im)};
}

// ------------------------------------------------------------------ MFMA wrappers (gfx950)
typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// D(16x16) += A(16x4) B(4x16). Lane l supplies A[l%16][l/16] and B[l/16][l%16]; accumulator
// element r of lane l is D[acc_row<R>(l/16, r)][l%16]. The row maps were measured with the
// probe kernel (afq_probe_mfma): FP64 holds rows g, g+4, g+8, g+12; FP32 holds rows 4g..4g+3.
__device__ inline d4 mfma16x16x4(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ inline f4 mfma16x16x4(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// D(16x16, f32) += A(16x32, bf16) B(32x16, bf16): lane l supplies A[l%16][8(l/16)+q] and
// B[8(l/16)+q][l%16], q = 0..7; the accumulator follows the FP32 layout (acc_row<float>).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
__device__ inline f4 mfma_bf16(bf16x8 a, bf16x8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

template <typename R> __host__ __device__ inline int acc_row(int g, int r);
template <> __host__ __device__ inline int acc_row<double>(int g, int r) { return 4 * r + g; }
template <> __host__ __device__ inline int acc_row<float>(int g, int r) { return 4 * g + r; }

template <typename R> struct acc_of;
template <> struct acc_of<double> { typedef d4 type; };
template <> struct acc_of<float> { typedef f4 type; };

// v plus the value of the lane `shift` below in the same row of 16 lanes (0 below the row)
template <int SHIFT>
__device__ inline double add_row_shr(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_update_dpp(0u, (unsigned)u, 0x110 + SHIFT, 0xf, 0xf, true);
  const unsigned hi =
      __builtin_amdgcn_update_dpp(0u, (unsigned)(u >> 32), 0x110 + SHIFT, 0xf, 0xf, true);
  return v + __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// lane 15 of each row of 16 lanes receives the sum of the row (DPP row shifts, no LDS)
__device__ inline double row_sum16(double v) {
  v = add_row_shr<1>(v);
  v = add_row_shr<2>(v);
  v = add_row_shr<4>(v);
  return add_row_shr<8>(v);
}

// ------------------------------------------------------------------ engine state
struct Workspace {
  int cap = 0;
  double* G = nullptr;       // c128 [W][N][M]
  double* X = nullptr;       // c128 [W][K]
  double* V = nullptr;       // c128 [W][M][M]
  double* HW = nullptr;      // c128 [W]
  double* mf = nullptr;      // c128 [W]
  double* ov = nullptr;      // c128 [W]
  double* E = nullptr;       // c128 [W][3]
  double* Kl = nullptr;      // c128 [W][K]
  double* exx = nullptr;     // c128 [W][nchunk]
  double* cum = nullptr;     // f64 [W]   population control: cumulative |w|
  int* off = nullptr;        // i32 [W]   offspring counts
  int* src = nullptr;        // i32 [W]   source walker of each slot (-1 = keep)
  int* ok = nullptr;         // i32 [1]   comb accepted the population
  double* split = nullptr;   // c128 [kMaxSplits][W][K]   split-k partials of vbias
  long split_elems = 0;
  double* esplit = nullptr;  // c128 split-k partials of the energy's traces (energy and vbias calls of one
  long esplit_elems = 0;     // handle may run on two streams)
};

// Region timers of a step (the AFQMCTimers regions of AFQMCTimer.h:25-63), as HIP events
// recorded on the launch stream around each region; read back (and summed) on demand.
enum Region {
  R_G_FOR_VBIAS = 0, R_VBIAS, R_ASSEMBLE_X, R_VHS, R_PROPAGATE, R_OVERLAP_G_E1, R_EXCHANGE,
  R_WALKER_UPDATE, R_ORTHO, R_COUNT
};
struct Timers {
  bool on = false;
  int cap = 0, used = 0;
  std::vector<hipEvent_t> ev;      // 2 per record
  std::vector<int> region;         // region of record i
  double ms[R_COUNT] = {0};
  long long count[R_COUNT] = {0};
};
// RAII region scope: records start/stop events when the timers are on.
struct RegionScope {
  Timers& t;
  hipStream_t s;
  int rec = -1;
  RegionScope(Timers& t_, hipStream_t s_, int r);
  ~RegionScope();
};

}  // namespace afq

struct afq_ham_s {
  int M = 0, N = 0, K = 0, walker_type = AFQ_CLOSED;
  double dt = 0.005, E0 = 0.0;
  double ci0_re = 1.0, ci0_im = 0.0;
  int precision = AFQ_FP64;
  int energy_route = AFQ_ROUTE_AUTO;
  int cfg_vbias = 0, cfg_vhs = 0, cfg_vhs_step = 0;   // GEMM tilings (afq_autotune): vbias, afq_vhs, a step's vHS
  afq_step_params params;
  int device = 0;
  // device tensors (built on the GPU at create)
  double* PsiT = nullptr;    // c128 [N][M]
  double* haj = nullptr;     // c128 [N][M]
  double* Lnak = nullptr;    // c128 [K][N][M]
  double* Likn = nullptr;    // f64 [M*M][K]
  double* h = nullptr;       // f64 [M][M]
  double* v0 = nullptr;      // f64 [M][M]
  double* vMF = nullptr;     // c128 [K]
  double* P1 = nullptr;      // c128 [M][M]
  double* H1 = nullptr;      // c128 [M][M]
  bool real_trial = false;   // every imaginary part of PsiT is zero (so is Im Lnak)
  bool sym = false;          // Likn[i][j] == Likn[j][i]: V_w is symmetric and kept as a triangle
  double* P1r = nullptr;     // f64 [2][M][M]: P1 and its transpose, when P1 is real
  bool P1_real = false;
  double* Lvb_d = nullptr;   // f64 [K][N*M padded to 16]: real Lnak rows (vbias of a real trial)
  float* Lvb_f = nullptr;    // f32 copy
  double* pairs = nullptr;   // f64 [re(, im)][N*M][N*M padded to 16]: pair table of the exchange (may be absent)
  double* Lp_d = nullptr;    // f64 [M(M+1)/2][K padded to 16]: rows i <= j of Likn (symmetric vHS)
  float* Lp_f = nullptr;     // f32 copy
  double* Lnak_r = nullptr;  // f64 [K][N][M padded to 16]: Re Lnak, only with a real trial
  float* Lnak_f = nullptr;   // c64 [K][N][M]   (FP32 contraction copies)
  float* Likn_f = nullptr;   // f32 [M*M][K]
  __bf16* Lnak_b = nullptr;  // bf16 [6 planes][K][16 NT][32 KC]  (BF16X3 exchange)
  __bf16* Lnak_g = nullptr;  // bf16 [6 planes][K][N*M padded to 32]   (BF16X3 vbias)
  __bf16* Likn_g = nullptr;  // bf16 [2 planes][M*M][K padded to 32]   (BF16X3 vHS)
  int8_t* Lnak_q = nullptr;  // i8 [6 slices][re(, im)][K][N][Mp] (INT8_SPLIT exchange)
  double* Lnak_u = nullptr;  // f64 [K][N]   power-of-two unit of each Lnak row
  int* Lnak_ord = nullptr;   // i32 [K]      slice-product order of each vector
  // [7]: eloc total/upper/lower, weight total/upper, population control calls/collapses
  unsigned long long* stats = nullptr;
  // back-propagation: the caller's field ring [fields_W][nfields][K] c128 and its position
  double* fields = nullptr;
  int nfields = 0, fields_W = 0;
  // weight factors and weight history [fields_W][3 nfields] c128 (caller-owned; null = none)
  double* wfac = nullptr;
  double* whis = nullptr;
  int* hist_pos = nullptr;   // device int
  double* P1H = nullptr;     // c128 [M][M]
  double* bp_ldet = nullptr; // c128 [bp_cap]
  int bp_cap = 0;
  afq::Workspace ws;
  afq::Timers timers;
};

namespace afq {

// Raises a kernel's dynamic-LDS limit to `bytes` (when above 64 KB) once per device. The
// attribute call is not a stream operation; doing it once keeps it out of every later launch,
// including launches recorded into a graph.
void ensure_dynamic_lds(const void* kern, size_t bytes);

// ------------------------------------------------------------------ launchers
// k_green.hip
void launch_green(hipStream_t s, int nb, int M, int N, const double* PsiT, const double* Phi,
                  long ldw, double* G, double* ov, int ov_mode, double ov_scale, cd ov_add,
                  const double* haj, double E0, double e1_scale, double* E, long ldE);
// k_gemm.hip:  C[m][n] = alpha * sum_k A[m][k] B[n][k]; A complex, B complex or real.
// split_ws (c128, split_ws_elems complex numbers) enables a deterministic split of k; NULL = none.
constexpr int kMaxSplits = 8;
int gemm_splits(int m, int n, int k);
// estimated us of launch_gemm_nt_z in FP64 with a complex B (two workgroups share a CU's rate, one alone
// reaches 0.6 of it, and the pass over the splits)
double gemm_nt_z_f64_us(int m, int n, int k, long split_elems);
// tilings launch_gemm_nt_z can run for a precision and kind of B (the cfg argument: 0 .. n-1)
int gemm_tile_configs(int precision, bool b_complex);
void launch_gemm_nt_z(hipStream_t s, int precision, int m, int n, int k, double alpha,
                      const double* A, long lda, const void* B, long ldb, bool b_complex,
                      double* C, long ldc, double* split_ws = nullptr, long split_ws_elems = 0,
                      int cfg = 0);
// k_gemm_real.hip: the same product with a real B, rows zero-padded to gemm_real_row(k) elements (f64
// for AFQ_FP64, else f32). nanmix: an Inf or NaN in A makes both parts of its row's sums NaN, as the
// zero imaginary part of a complex B does. FP32 gives launch_gemm_nt_z's bits.
int gemm_real_row(int k);
int gemm_real_tile_configs(int precision);   // its tilings (cfg: 0 .. n-1)
// padded rows dst[row][0..gemm_real_row(k)) = src[row][0..k) (the real part of a complex src);
// packed_n > 0: the packed_n (packed_n + 1) / 2 rows i <= j of the n x n rows of src
void launch_pad_rows(hipStream_t s, long rows, int k, int packed_n, const double* src, bool complex_src,
                     double* dst);
void launch_pad_rows(hipStream_t s, long rows, int k, int packed_n, const double* src, bool complex_src,
                     float* dst);
void launch_gemm_real(hipStream_t s, int precision, int m, int n, int k, double alpha,
                      const double* A, long lda, const void* B, double* C, long ldc, bool nanmix,
                      double* split_ws = nullptr, long split_ws_elems = 0, int cfg = 0);
// k_gemm_real.hip: the exchange sum_n tr(T_n^2) as the quadratic form G B G^T of the flat rows
// G[w][(a, i)], B[(b, j)][(a, i)] = sum_n Lnak[n][b][i] Lnak[n][a][j] (upper triangle, off-diagonal
// entries doubled; a real and, unless Lnak is real, an imaginary table). L: Lnak (c128 [K][N M]) or its
// real rows of gemm_real_row(N M). At most max_parts partials per walker (1 + (N M - 1) / 64 per table
// are always possible).
size_t pair_table_elems(int NM, bool real);
void launch_pair_table(hipStream_t s, int M, int N, int K, const double* L, bool real, double* B);
int pair_parts(int W, int NM, bool real, int max_parts);
void launch_pair_exchange(hipStream_t s, int W, int NM, bool real, int max_parts, const double* G,
                          const double* B, double* part);
// the work of launch_pair_exchange's fullest CU (rows of its tiles times their mean k), and estimated us of
// launch_gemm_real in FP64
double pair_exchange_cost(int W, int NM, bool real, int max_parts);
double gemm_f64_us(int m, int n, int k, long split_elems);
// k_energy.hip
int device_cus();                        // compute units of the current device (cached)
int exx_nchunks(int W, int N, int K);   // chunks of Cholesky vectors the exchange kernel uses
double exchange_general_us(int precision, int W, int M, int N, int K);   // estimated us of launch_exchange
// k_exchange_f64.hip: the exchange of the FP64 form on up to 128 orbitals; Lreal (may be NULL) is
// the zero-padded real Lnak of a real trial
bool exchange_f64_supported(int M, int N);
int exchange_f64_chunks(int W, int N, int K);   // tr(T^2) partials per walker
double exchange_f64_us(int W, int M, int N, int K, bool real);   // estimated us of launch_exchange_f64
int real_lnak_row(int M);                       // padded row length of Lreal
void launch_exchange_f64(hipStream_t s, int W, int M, int N, int K, const double* G,
                         const double* Lnak, const double* Lreal, double* Kl, double* part);
void launch_split_reduce(hipStream_t s, int m, int n, int splits, double alpha,
                         const double* split_ws, double* C, long ldc);
// k_gemm_bf16.hip: the BF16X3 form of the Cholesky GEMMs (three-product complex multiplication,
// hi/lo BF16 splits, FP32 accumulation); B as BF16 planes from split_planes_bf16 (complex: 6
// planes, real: 2, rows padded to bf16_row(cols))
int bf16_row(int cols);
void split_planes_bf16(hipStream_t s, long rows, int cols, bool complex_src, const double* src,
                       __bf16* dst);
void launch_gemm_bf16(hipStream_t s, int m, int n, int k, double alpha, const double* A, long lda,
                      const __bf16* Bp, bool b_complex, double* C, long ldc,
                      double* split_ws = nullptr, long split_ws_elems = 0);
// k_exchange_bf16.hip: the exchange in the BF16X3 form (N <= 32, M <= 128)
bool exchange_bf16_supported(int M, int N);
size_t exchange_bf16_elems(int M, int N, int K);   // bf16 elements of the exchange planes
int exchange_bf16_chunk(int W, int N, int K);
int exchange_bf16_chunks(int W, int N, int K);
double exchange_bf16_us(int W, int M, int N, int K);   // estimated us of launch_exchange_bf16
void split_lnak_bf16(hipStream_t s, int M, int N, int K, const double* Lnak, __bf16* Lb);
void launch_exchange_bf16(hipStream_t s, int W, int M, int N, int K, const double* G,
                          const __bf16* Lb, double* Kl, double* exx_part);
// k_exchange_i8.hip: the exchange on int8 MFMA, Ozaki-split rows (N <= 32, M <= 128); real: Im Lnak
// is zero and only its real slices are kept
bool exchange_i8_supported(int M, int N);
int exchange_i8_row(int M);                                // Mp: padded row length of the slices
size_t exchange_i8_bytes(int M, int N, int K, bool real);  // size of the Lnak slices
int exchange_i8_chunks(int W, int M, int N, int K, bool real);   // tr(T^2) partials per walker
void split_lnak_i8(hipStream_t s, int M, int N, int K, const double* Lnak, bool real, int8_t* Lq,
                   double* Lu);
// per Cholesky vector the slice-product order (set-up, synchronous)
void exchange_i8_check(int M, int N, int K);   // AFQ_EUNSUPPORTED for shapes that the int8 form refuses
void exchange_i8_orders(hipStream_t s, int M, int N, int K, const double* Lnak, int* ord);
void launch_exchange_i8(hipStream_t s, int W, int M, int N, int K, const double* G, bool real,
                        const int8_t* Lq, const double* Lu, const int* ord, double* Kl,
                        double* exx_part);
// k_exchange_i8w.hip: the same per walker (17 to 32 electrons: complex trials on more than 64 orbitals)
int exchange_i8w_chunks(int W, int N, int K);
void launch_exchange_i8w(hipStream_t s, int W, int M, int N, int K, const double* G, bool real,
                         const int8_t* Lq, const double* Lu, const int* ord, double* Kl, double* exx_part);
void launch_exchange(hipStream_t s, int precision, int W, int M, int N, int K, const double* G,
                     const void* Lnak, double* Kl, double* exx_part);
void launch_energy_finalize(hipStream_t s, int W, int K, int nchunk, int walker_type,
                            const double* Kl, const double* exx_part, double* E);
void launch_e1(hipStream_t s, int W, int M, int N, const double* G, const double* haj,
               double E0, double scl, double* E);
// k_propagate.hip
enum class VKind {
  full,          // V_w [M][M]
  packed,        // its upper triangle, row by row (symmetric V)
  packed_adjoint // the same, applied as -V^H
};
// P1r: the real P1 as f64 [M][M], NULL when P1 is complex
void launch_propagate(hipStream_t s, int nb, int M, int N, double* Phi, long ldw,
                      const double* P1, const double* P1r, const double* V, VKind kind, int order);
// k_qr.hip
void launch_orthogonalize(hipStream_t s, int nb, int M, int N, double* Phi, long ldw,
                          double* logdetR);
// k_walker.hip
void launch_store_fields(hipStream_t s, int W, int K, const double* X, double* ring, int nfields,
                         const int* pos);
void launch_advance_history(hipStream_t s, int* pos, int nhist);
void launch_neg_adjoint(hipStream_t s, int W, int M, double* V);
void launch_adjoint(hipStream_t s, int M, const double* A, double* B);
void launch_add_strided(hipStream_t s, int W, const double* x, double* out, long stride);
void launch_construct_X(hipStream_t s, int W, int K, double vbias_bound, int project,
                        int free_projection, const double* vMF, const double* xi, double* X,
                        double* HW, double* mf);
void launch_walker_update(hipStream_t s, int W, double* wbuf, long ldw, long poff,
                          const afq_step_params& p, double dt, double Eshift, double E0,
                          const double* ov, const double* E, const double* mf,
                          const double* HW, int hybrid, unsigned long long* stats,
                          double* wfac = nullptr, double* whis = nullptr, int nhist = 0,
                          const int* pos = nullptr);
void launch_set_properties(hipStream_t s, int W, double* wbuf, long ldw, long poff,
                           const double* ov, const double* E, int seed_pseudo);
void launch_weighted_sums(hipStream_t s, int W, const double* wbuf, long ldw, long poff,
                          double dt, double* out);
void launch_estimator_sums(hipStream_t s, int W, const double* wbuf, long ldw, long poff,
                           double dt, const double* E, const double* ov, double* out);
void launch_probe_mfma(hipStream_t s, int kind, double* out);
// the per-walker back-propagation rows that population control moves with the walkers: the
// field ring [W][fields_ld] c128 and the weight-factor / weight-history rings [W][nhist] c128
// (null when absent), and the history position on the device
struct BackPropRows {
  double* fields = nullptr;
  long fields_ld = 0;
  double* wfac = nullptr;
  double* whis = nullptr;
  int nhist = 0;
  const int* pos = nullptr;
};
void launch_population_control(hipStream_t s, int W, double* wbuf, long ldw, long poff,
                               double r, double* cum, int* off, int* src, int* ok,
                               unsigned long long* stats, const BackPropRows* bp = nullptr);
// k_setup.hip
void setup_hamiltonian(afq_ham_s* H, hipStream_t s);
void launch_v0(hipStream_t s, int M, int K, const double* Likn, double* v0);
// whether L[i][j][n] equals L[j][i][n] bit for bit for all i, j, n (synchronises the stream)
bool likn_symmetric(hipStream_t s, int M, int K, const double* Likn);
// dst[row][0..ld) = Re src[row][0..M), zero-padded
void launch_real_rows(hipStream_t s, long rows, int M, int ld, const double* src, double* dst);
void launch_zero_imag(hipStream_t s, int n, double* v);
// P1 [M][M] c128 on the host as the reference applies it: |x| <= 1e-8 dropped, imaginary
// roundoff dropped when P1 is real to 1e-14
void sparsify_one_body_propagator(int M, double* P);
void build_one_body_propagator(hipStream_t s, int M, int K, double dt, const double* h,
                               const double* v0, const double* Likn, const double* vMF,
                               double* H1, double* P1, double* P1r, bool* real);
// k_phmsd.hip
// ws: ph_2body_workspace() doubles for the staged kernel (NULL or too small: the per-walker one)
long ph_2body_workspace(int nw, int nact, int nelec, int nchol);
void launch_ph_2body(hipStream_t s, int nw, int ndet, int nex, int nact, int nelec, int nchol,
                     const int* iexcit, const int* refc, const double* Twina, const double* R,
                     const double* wgt, double* EX, double* EJ, double* KE,
                     double* ws = nullptr, long ws_doubles = 0);
void launch_ph_1body(hipStream_t s, int nw, int ndet, int nex, int nact, int nelec,
                     const int* iexcit, const int* refc, const double* S, const double* R,
                     const double* wgt, double* E);
void launch_ph_woodbury(hipStream_t s, int nb, int nmo, int nel, int nact, const double* A,
                        const int* ref, const double* Phi, long ldw, double* G, double* ov,
                        double* QQ0, double* work);
// the same with the reference at orbitals 0..nel-1 (A's first nel rows)
void launch_ph_reference_G(hipStream_t s, int nb, int nmo, int nel, int nact, const double* A,
                           const double* Aref, const double* Phi, long ldw, double* G, double* ov,
                           double* QQ0);
void launch_ph_spin_weights(hipStream_t s, int nw, int nu, const int* cp, const int* ci,
                            const double* cv, const double* rup, const double* rdn, double* wgt,
                            double* ov);
void launch_ph_overlaps(hipStream_t s, int nw, int ndet, int nex, int nact, int nelec,
                        const int* iexcit, const double* T, double* ov);
void launch_ph_compact_R(hipStream_t s, int nw, int ndet, int nex, int nact, int nelec,
                         const int* iexcit, const int* refc, const double* T, double* R);
void launch_ph_reference_energy(hipStream_t s, int nw, int nel, int nmo, int nchol, int nact,
                                double scl, double E0, const double* G, const double* Lna,
                                const double* haj, double* E, double* Kl, double* Twina,
                                double* Swia);
void launch_ph_couple_ke(hipStream_t s, int nw, int nchol, int nout, const int* cp, const int* ci,
                         const double* cv, const double* rin, const double* KEin,
                         const double* rout, double* KEout);
void launch_ph_ke_dot(hipStream_t s, int nw, int nchol, int nd, const double* a, const double* b,
                      double* out, int ostride);
void launch_ph_accumulate(hipStream_t s, int nw, const double* Eref, const double* Ov,
                          const double* Ex, double* acc);
void launch_ph_finalize(hipStream_t s, int nw, const double* acc, const double* Ov,
                        const double* log_ov, double* E, double* ov_out);
void launch_ph_fill(hipStream_t s, long n, double re, double im, double* x);
void launch_ph_rg(hipStream_t s, int nw, int nel, int nact, int nmo, int ldrows, int row0,
                  const double* R, const double* GA, const double* Ov, double* G);
void launch_ph_full_g(hipStream_t s, int nw, int nact, int nmo, const double* A0,
                      const double* A1, const double* Gc, double* Gf);
void launch_ph_log_overlap(hipStream_t s, int nw, const double* Ov, const double* log_ov,
                           double* out);
void launch_ph0_products(hipStream_t s, int nw, int nmo, int nel, int nact, int nchol,
                         const double* Phi, long ldw, const double* A, const double* haj,
                         const double* Lna, bool lna_complex, double* Phit, double* TAB,
                         double* Hp, double* P);
void launch_ph0_config(hipStream_t s, int nw, int nc, int nel, int nact, int nchol,
                       const int* conf, const double* TAB, const double* Hp, const double* P,
                       double E0, double* ld, double* Emsd, double* KE, const double* KEr,
                       double* Tinv);
void launch_ph0_ratios(hipStream_t s, int nw, int nc, double* r, double* log_ov);
void launch_ph0_assemble(hipStream_t s, int nw, int nu, int nd, const double* wgt0,
                         const double* Em0, const double* wgt1, const double* Em1,
                         const double* r1, double* acc);
// k_phmsd_exc.hip: an expansion's excited determinants as rank-nex corrections of the reference
// (the reference determinant at orbitals 0..nel-1, every particle at nel or above)
struct PhShell {
  int nex, ndet, row;   // rank, determinants, first row of the ratio and weight arrays
  int qoff;             // first element of the shell's Q per walker: Q[w][qoff + (e nex + q) ndet + d]
  const int* iexcit;    // device [ndet][2 nex]
};
int ph_exc_vectors(int nel, int nact);               // vectors per workgroup; 0: not supported
int ph_exc_groups(int nel, int nact, int nchol);     // groups of vectors (8 complex sums each)
void launch_ph_ratios_q(hipStream_t s, int nw, int nel, int nact, long qtot, int nshell, int maxdet,
                        int maxnex, const PhShell* shells, const double* QQ0, double* ratio,
                        double* Q);
void launch_ph_weights(hipStream_t s, int nw, int nu, const int* cp, const int* ci,
                       const double* cv, const double* own, const double* other, double* wgt,
                       double* sum);
void launch_ph_exc(hipStream_t s, bool down, int nw, int nel, int nact, int nchol, long qtot,
                   int nshell, int maxnex, int nu_own, int nu_up, const PhShell* shells,
                   const double* T, const double* QQ0, const double* Q, const double* wgt,
                   double* KE, const int* cp, const int* ci, const double* cv, const double* rup,
                   const double* rdn, double* part);
void launch_ph_exc_finish(hipStream_t s, int nw, int nu, int gu, int gd, double E0, const double* wgt,
                          const double* pu, const double* pd, const double* log_ov, double* E,
                          double* ov);
void launch_ph_expansion_R(hipStream_t s, int nw, int nel, int nact, int nu, long qtot,
                           const int* rp, const int* ru, const int* rq, const double* QQ0,
                           const double* Q, const double* wgt, double* R, double* ov);
void launch_ph_density(hipStream_t s, int nw, int nup, int ndn, int nact, int nmo, bool fold,
                       const double* R0, const double* A0, const double* G0, const double* R1,
                       const double* A1, const double* G1, const double* ov, double* U0, double* U1,
                       double* F);
void launch_ph_rows_of_vectors(hipStream_t s, int nmo, int nchol, bool fold, int ld,
                               const double* Likn, double* out);
void launch_ph_accumulate_R(hipStream_t s, int nw, int ndet, int nex, int nact, int nelec,
                            const int* iexcit, const int* refc, const double* Rc,
                            const double* ov, const double* wgt, double* R);

}  // namespace afq
