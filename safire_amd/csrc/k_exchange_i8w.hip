// The exchange on int8 MFMA (k_exchange_i8.hip has the slices, the orders and the rule between the two) with
// the tiles of a walker by themselves: one 16 x 16 tile of T per walker and vector for up to 16 electrons,
// 2 x 2 for 17 to 32.
//
// Against the product packed across walkers and vectors, rows and columns are padded to 16 or 32, but
// nothing else is shared: up to 16 electrons every wavefront goes from its MFMAs to the sums of its own T
// without a barrier over the workgroup, and a 2 x 2 tile of complex products leaves registers for two
// wavefronts per SIMD. So it is taken where padding costs little, and in small calls. Energies in us, packed
// and here (M, N, K, walkers): real trial 24, 6, 36, 64 20 and 17; 64, 16, 96, 256 45 and 34; 128, 16, 192,
// 256 99 and 84; 64, 8, 320, 1024 98 and 229. Complex trial 64, 16, 96, 256 54 and 44; 128, 16, 640, 1024
// 1699 and 1496; 128, 32, 64, 1024 660 and 435; 128, 32, 640, 1024 6140 and 3850; 77, 19, 385, 1024 1910 and
// 2250.
#include "i8_split.hpp"

#include <algorithm>

namespace afq {

namespace {

using namespace i8;

// ---- up to 16 electrons: four walkers (wavefronts) per workgroup, two workgroups per CU, so that one's
// FP64 sums run under the other's MFMAs. Each wavefront slices its walker's G once; the slices of kStage
// vectors at a time go through LDS, double-buffered; each T block goes through the wavefront's LDS.
constexpr int kWPB = 4;

// vectors staged together: two, or one where a vector is 27 KB (complex Lnak on more than 64 orbitals)
template <int KC, bool LC>
constexpr int kStageOf = KC == 2 && LC ? 1 : 2;

// orders LDS traffic of one wavefront: its own writes are visible to its own later reads
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int KC, int NV, bool LC>
__global__ __launch_bounds__(64 * kWPB, 2) void k_exchange_i8_w1(
    int W, int M, int N, int K, int Mp, int kChunk, const double* __restrict__ G,
    const int8_t* __restrict__ Lq, const double* __restrict__ Lu, const int* __restrict__ ord,
    double* __restrict__ Kl, double* __restrict__ exx_part, int nchunk) {
  constexpr int NP = LC ? 2 : 1;
  constexpr int kStage = kStageOf<KC, LC>;
  constexpr int ROWB = 64 * KC + 16;             // staged row (bytes): the row plus 16 of padding
  constexpr int kCombos = kStage * kS * NP;      // (vector, slice, part)
  constexpr int kPiece = 16 * 4 * KC;            // 16-byte pieces of one of them
  constexpr int kPre = (kCombos * kPiece + 64 * kWPB - 1) / (64 * kWPB);
  static_assert((64 * kWPB) % kPiece == 0, "staging positions must tile the workgroup");
  __shared__ __attribute__((aligned(16))) int8_t sBuf[2][kCombos * 16 * ROWB];
  __shared__ double sUnit[2][kStage][16];        // column units of the staged vectors
  // per-wavefront T block [a][b], rows padded to 17 entries: distinct banks down a column
  __shared__ __attribute__((aligned(16))) double2 sT[kWPB][16 * 17];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = tid >> 6;
  const int g = lane >> 4, r16 = lane & 15;
  const int w_raw = blockIdx.x * kWPB + wave;
  const bool active = w_raw < W;
  const int w = active ? w_raw : W - 1;
  const int c = blockIdx.y;
  const int nbeg = c * kChunk, nend = min(K, nbeg + kChunk);
  const size_t plane = (size_t)K * N * Mp;       // bytes of one slice of one part
  const int NMp = N * Mp;

  i4 ar[KC][kS], ai[KC][kS];
  const double uG = slice_row<KC>(reinterpret_cast<const double2*>(G) + ((long)w * N + min(r16, N - 1)) * M,
                                  r16 < N, M, g, ar, ai);
  double uRow[4];   // units of the accumulator rows, over 254: the joined orders carry a factor 254
#pragma unroll
  for (int r = 0; r < 4; ++r) uRow[r] = __shfl(uG, 4 * g + r, 64) * (1.0 / kBase);

  // Slot i of a thread is (row, 16-byte column), the same in all of its slots, and (vector, slice, part),
  // the same over a wavefront
  const int pos = tid % kPiece;
  const int pb = pos / (4 * KC), pkv = pos % (4 * KC);
  const bool pos_ok = pb < N && 16 * pkv < Mp;
  const int gpos = pb * Mp + 16 * pkv, lpos = pb * ROWB + 16 * pkv;
  uint4 pre[kPre];
  double preU = 0.0;
  auto load_group = [&](int nv0) {
#pragma unroll
    for (int i = 0; i < kPre; ++i) {
      const int combo = __builtin_amdgcn_readfirstlane((i * 64 * kWPB + tid) / kPiece);
      const int v = combo / (kS * NP), tp = combo - v * (kS * NP);
      pre[i] = uint4{0u, 0u, 0u, 0u};
      if (combo < kCombos && nv0 + v < nend && pos_ok)
        pre[i] = *reinterpret_cast<const uint4*>(Lq + tp * plane + (size_t)(nv0 + v) * NMp + gpos);
    }
    if (tid < kStage * 16) {
      const int v = tid / 16, b = tid % 16, n = nv0 + v;
      preU = (n < nend && b < N) ? Lu[(long)n * N + b] : 0.0;
    }
  };
  auto store_group = [&](int buf) {
#pragma unroll
    for (int i = 0; i < kPre; ++i) {
      const int combo = __builtin_amdgcn_readfirstlane((i * 64 * kWPB + tid) / kPiece);
      if (combo < kCombos) *reinterpret_cast<uint4*>(sBuf[buf] + combo * 16 * ROWB + lpos) = pre[i];
    }
    if (tid < kStage * 16) sUnit[buf][tid / 16][tid % 16] = preU;
  };

  double exx_re = 0.0, exx_im = 0.0;
  double2* T = sT[wave];
  // NV vectors from staged vector h on, with the slice products s + t <= ON
  auto vectors = [&](auto on_c, int nv0, int h, const int8_t* sB, const double (*sU)[16]) {
    constexpr int ON = decltype(on_c)::value;
    i4 cR[NV][ON + 1], cI[NV][ON + 1], cQ[NV][LC ? ON + 1 : 1];
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int o = 0; o <= ON; ++o) {
        cR[v][o] = i4{0, 0, 0, 0};
        cI[v][o] = i4{0, 0, 0, 0};
        if (LC) cQ[v][LC ? o : 0] = i4{0, 0, 0, 0};
      }
#pragma unroll
    for (int kc = 0; kc < KC; ++kc)
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int t = 0; t <= ON; ++t) {
          const int8_t* base = sB + (((h + v) * kS + t) * NP * 16 + r16) * ROWB + 64 * kc + 16 * g;
          const i4 br = *reinterpret_cast<const i4*>(base);
          const i4 bi = LC ? *reinterpret_cast<const i4*>(base + 16 * ROWB) : br;
#pragma unroll
          for (int s = 0; s + t <= ON; ++s) {
            cR[v][s + t] = mfma_i8(ar[kc][s], br, cR[v][s + t]);
            cI[v][s + t] = mfma_i8(ai[kc][s], br, cI[v][s + t]);
            if (LC) {
              cQ[v][LC ? s + t : 0] = mfma_i8(ai[kc][s], bi, cQ[v][LC ? s + t : 0]);
              cI[v][s + t] = mfma_i8(ar[kc][s], bi, cI[v][s + t]);
            }
          }
        }
    // T block -> LDS, tr(T^2) lane partials, tr(T) -> Kl
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int n = nv0 + h + v;
      const double uL = sU[h + v][r16];
      if (LC)
#pragma unroll
        for (int o = 0; o <= ON; ++o) cR[v][o] -= cQ[v][LC ? o : 0];
      double2 x[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double u = uRow[r] * uL;
        x[r] = double2{join_orders<ON, KC, LC>(cR[v], r) * u, join_orders<ON, KC, LC>(cI[v], r) * u};
      }
      wave_lds_sync();
#pragma unroll
      for (int r = 0; r < 4; ++r) T[(4 * g + r) * 17 + r16] = x[r];
      wave_lds_sync();
      if (n < nend) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const double2 y = T[r16 * 17 + 4 * g + r];
          exx_re += x[r].x * y.x - x[r].y * y.y;
          exx_im += x[r].x * y.y + x[r].y * y.x;
        }
        // tr(T): the N diagonal entries in lanes 0..15, summed into lane 15 by DPP row shifts
        double2 d = double2{0.0, 0.0};
        if (lane < N) d = T[lane * 17 + lane];
        const double dr = row_sum16(d.x), di = row_sum16(d.y);
        if (lane == 15 && active)
          *reinterpret_cast<double2*>(Kl + 2 * ((long)w * K + n)) = double2{dr, di};
      }
    }
  };

  if (nbeg < nend) {
    load_group(nbeg);
    store_group(0);
  }
  __syncthreads();
  for (int nv0 = nbeg, buf = 0; nv0 < nend; nv0 += kStage, buf ^= 1) {
    const bool more = nv0 + kStage < nend;
    if (more) load_group(nv0 + kStage);   // in flight during this group's MFMAs
    int on = ord[nv0];
    if (kStage > 1) on = max(on, ord[min(nv0 + 1, nend - 1)]);
    on = __builtin_amdgcn_readfirstlane(on);
#pragma unroll 1
    for (int h = 0; h < kStage; h += NV) {
      if (on > 4) vectors(std::integral_constant<int, 5>(), nv0, h, sBuf[buf], sUnit[buf]);
      else vectors(std::integral_constant<int, 4>(), nv0, h, sBuf[buf], sUnit[buf]);
    }
    // the other buffer was last read in the previous group, before the barrier that ended it
    if (more) store_group(buf ^ 1);
    __syncthreads();
  }

  for (int off = 32; off > 0; off >>= 1) {
    exx_re += __shfl_xor(exx_re, off, 64);
    exx_im += __shfl_xor(exx_im, off, 64);
  }
  if (lane == 0 && active)
    *reinterpret_cast<double2*>(exx_part + 2 * ((long)w * nchunk + c)) = double2{exx_re, exx_im};
}

// ---- 17 to 32 electrons, complex Lnak on 65 to 128 orbitals: T_wn is 2 x 2 tiles. An 8-wavefront workgroup holds 4 walkers; the two wavefronts
// of a walker own its row tiles ta = 0, 1 and compute both column tiles of their rows.
//
// tr(T^2) = tr(T00^2) + tr(T11^2) + 2 tr(T01 T10): wavefront ta = 0 takes the first and the cross
// term (it holds T01 in registers and reads T00^T and T10 from LDS), wavefront 1 the second; so only T00,
// T10 and T11 go to LDS, and wavefront 0 takes tr(T) from their diagonals. The two row tiles write
// separate tr(T^2) partials (slots 2c and 2c + 1 of the walker).
//
// Staging: the slices of one vector (12 slice-parts x 32 rows x 128 bytes) are copied from global
// memory straight into LDS, double-buffered in two LDS objects with the vector loop unrolled by two:
// every access names its buffer statically, so the compiler does not wait for the next vector's copies
// before reading the current one. Rows are not padded; the 16-byte piece kv of row b sits at position
// kv ^ f(b) of its row, which spreads the 16 rows an MFMA fragment reads over distinct banks. Rows
// b >= N and pieces past the end of a row copy clamped (in-bounds) data: their column unit is 0 and the
// matching G entries are 0.
constexpr int kT2Walkers = 4;

__device__ inline int t2_swz(int b) { return (b >> 1) & 7; }

__device__ inline double readlane_d(double v, int lane) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, lane);
  const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), lane);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

__global__ __launch_bounds__(128 * kT2Walkers, 2) void k_exchange_i8_w2(
    int W, int M, int N, int K, int Mp, int kChunk, const double* __restrict__ G,
    const int8_t* __restrict__ Lq, const double* __restrict__ Lu, const int* __restrict__ ord,
    double* __restrict__ Kl, double* __restrict__ exx_part, int nslots) {
  constexpr int KC = 2, NP = 2;
  constexpr int kRows = 32;
  constexpr int ROWB = 64 * KC;                  // staged row (bytes), unpadded
  constexpr int kPlane = kRows * ROWB;           // one slice-part of one vector
  constexpr int kVecBytes = kS * NP * kPlane;
  constexpr int kWindows = kVecBytes / 1024;     // 1 KB copied per wavefront instruction
  constexpr int kWaves = 2 * kT2Walkers;
  constexpr int kTile = 16 * 16;
  static_assert(kVecBytes % 1024 == 0, "a vector's slices are whole 1 KB windows");
  __shared__ __attribute__((aligned(16))) int8_t sB0[kVecBytes];
  __shared__ __attribute__((aligned(16))) int8_t sB1[kVecBytes];
  __shared__ double sU0[kRows];
  __shared__ double sU1[kRows];
  // per walker the tiles T00, T10, T11 [x][y]; entry (x, y) sits in column y ^ x of row x, so that 16
  // lanes reading down a column hit 16 different banks
  __shared__ __attribute__((aligned(16))) double2 sT[kT2Walkers][3 * kTile];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int g = lane >> 4, r16 = lane & 15;
  const int wl = wave >> 1, ta = wave & 1;
  const int w_raw = blockIdx.x * kT2Walkers + wl;
  const bool active = w_raw < W;
  const int w = active ? w_raw : W - 1;
  const int c = blockIdx.y;
  const int nbeg = c * kChunk, nend = min(K, nbeg + kChunk);
  const size_t plane = (size_t)K * N * Mp;
  const int arow = ta * 16 + r16;                // this lane's row of G

  i4 ar[KC][kS], ai[KC][kS];
  const double uG = slice_row<KC>(reinterpret_cast<const double2*>(G) + ((long)w * N + min(arow, N - 1)) * M,
                                  arow < N, M, g, ar, ai);
  double uRow[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) uRow[r] = __shfl(uG, 4 * g + r, 64) * (1.0 / kBase);

  double exx_re = 0.0, exx_im = 0.0;
  double2* T = sT[wl];
  auto tpos = [](int x, int y) { return x * 16 + (y ^ x); };   // within a tile

  // copy vector n's slices into dst: lane l of window win writes bytes 1024 win + 16 l ..
  auto stage = [&](int n, int8_t* dst) {
    for (int win = wave; win < kWindows; win += kWaves) {
      const int o = win * 1024 + 16 * lane;
      const int tp = o / kPlane;
      const int b = (o % kPlane) / ROWB;
      const int kv = ((o % ROWB) >> 4) ^ t2_swz(b);
      const int bg = min(b, N - 1);
      const int kg = min(16 * kv, Mp - 16);
      const int8_t* src = Lq + tp * plane + ((size_t)n * N + bg) * Mp + kg;
      __builtin_amdgcn_global_load_lds(
          (const void __attribute__((address_space(1)))*)src,
          (void __attribute__((address_space(3)))*)(dst + win * 1024), 16, 0, 0);
    }
  };
  double preU = 0.0;
  auto load_units = [&](int n) {
    if (threadIdx.x < kRows) preU = (int)threadIdx.x < N ? Lu[(long)n * N + threadIdx.x] : 0.0;
  };

  if (nbeg < nend) {
    load_units(nbeg);
    stage(nbeg, sB0);
  }
  // one vector: its slices are in sBb (or in flight to it) and its column units in preU; they
  // go to uB here, and the next vector's slices to sBn
  auto vector = [&](int n, const int8_t* sBb, double* uB, int8_t* sBn) {
    // vector n is in sBb (this thread's copies done, then everyone's); every wavefront is past
    // vector n - 1, so sBn, uB and the T tiles are free again
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
    if (threadIdx.x < kRows) uB[threadIdx.x] = preU;
    __syncthreads();
    const int on = __builtin_amdgcn_readfirstlane(ord[n]);   // this vector's slice order
    if (n + 1 < nend) {
      load_units(n + 1);   // before the copies: waiting for it leaves them in flight
      stage(n + 1, sBn);
    }
    double2 k01[4];        // T01 (rows of wavefront 0, column tile 1) stays in registers
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      i4 acR[kS], acI[kS], acQ[kS];
#pragma unroll
      for (int o = 0; o < kS; ++o) {
        acR[o] = i4{0, 0, 0, 0};
        acI[o] = i4{0, 0, 0, 0};
        acQ[o] = i4{0, 0, 0, 0};
      }
      const int row = tb * 16 + r16;
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        const int chunk = (((4 * kc + g) ^ t2_swz(row)) << 4);
#pragma unroll
        for (int t = 0; t < kS; ++t) {
          if (t > on) break;   // uniform over the workgroup
          const int8_t* base = sBb + (t * NP * kRows + row) * ROWB + chunk;
          const i4 br = *reinterpret_cast<const i4*>(base);
          const i4 bi = *reinterpret_cast<const i4*>(base + kPlane);
#pragma unroll
          for (int s = 0; s < kS; ++s)
            if (s + t < kS && s + t <= on) {
              acR[s + t] = mfma_i8(ar[kc][s], br, acR[s + t]);
              acI[s + t] = mfma_i8(ar[kc][s], bi, acI[s + t]);
              acQ[s + t] = mfma_i8(ai[kc][s], bi, acQ[s + t]);
              acI[s + t] = mfma_i8(ai[kc][s], br, acI[s + t]);
            }
        }
      }
#pragma unroll
      for (int o = 0; o < kS; ++o) acR[o] -= acQ[o];
      const double uL = uB[row];
#pragma unroll
      for (int r = 0; r < 4; ++r) {   // orders past `on` are zero
        const double u = uRow[r] * uL;
        const double2 x = double2{join_orders<5, KC, true>(acR, r) * u, join_orders<5, KC, true>(acI, r) * u};
        if (ta == 0 && tb == 1) k01[r] = x;
        else T[(ta == 0 ? 0 : 1 + tb) * kTile + tpos(4 * g + r, r16)] = x;
      }
    }
    lds_barrier();   // T00, T10, T11 of every walker are in LDS
    // ta = 0: sum_{a,b in tile 0} T_ab T_ba + 2 sum_{a in 0, b in 1} T_ab T_ba;
    // ta = 1: sum_{a,b in tile 1} T_ab T_ba. For (a, b) = (4 g + r, r16) within the tiles, T_ab
    // is entry (4 g + r, r16) of its tile and T_ba entry (r16, 4 g + r) of the tile (row tile of
    // b, column tile of a).
    {
      const double2* diag = T + (ta == 0 ? 0 : 2) * kTile;   // T00 or T11
      const double2* cross = T + 1 * kTile;                 // T10
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int xx = 4 * g + r;
        const double2 x = diag[tpos(xx, r16)], y = diag[tpos(r16, xx)];
        exx_re += x.x * y.x - x.y * y.y;
        exx_im += x.x * y.y + x.y * y.x;
        if (ta == 0) {
          const double2 z = cross[tpos(r16, xx)];
          exx_re += 2.0 * (k01[r].x * z.x - k01[r].y * z.y);
          exx_im += 2.0 * (k01[r].x * z.y + k01[r].y * z.x);
        }
      }
    }
    if (ta == 0) {
      // tr(T): diagonals of T00 (lanes 0..15) and T11 (lanes 16..31), rows a < N
      double2 d = double2{0.0, 0.0};
      if (lane < N) d = T[(lane < 16 ? 0 : 2) * kTile + tpos(lane & 15, lane & 15)];
      const double dr = row_sum16(d.x), di = row_sum16(d.y);
      const double kr = readlane_d(dr, 15) + readlane_d(dr, 31);
      const double ki = readlane_d(di, 15) + readlane_d(di, 31);
      if (lane == 0 && active) *reinterpret_cast<double2*>(Kl + 2 * ((long)w * K + n)) = double2{kr, ki};
    }
  };
  for (int n = nbeg; n < nend; n += 2) {
    vector(n, sB0, sU0, sB1);
    if (n + 1 < nend) vector(n + 1, sB1, sU1, sB0);
  }

  for (int off = 32; off > 0; off >>= 1) {
    exx_re += __shfl_xor(exx_re, off, 64);
    exx_im += __shfl_xor(exx_im, off, 64);
  }
  if (lane == 0 && active)
    *reinterpret_cast<double2*>(exx_part + 2 * ((long)w * nslots + 2 * c + ta)) = double2{exx_re, exx_im};
}

// Vectors per workgroup: the multiple of the staging group that fills whole rounds of the resident
// workgroups best (two per CU up to 16 electrons, one above), the larger one of equals. 17 to 32
// electrons: two partials per walker and chunk, so chunks of at least 2 vectors keep them to K + 1, and
// the chunks may span all vectors (each of them reads and slices G again).
int chunk_of(int W, int N, int K) {
  const int step = 2;
  const int wpb = N > 16 ? kT2Walkers : kWPB;
  const long cus = device_cus() * (N > 16 ? 1L : 2L);
  const long wgroups = (W + wpb - 1) / wpb;
  const int jmax = N > 16 ? (K + step - 1) / step : 16;
  int best = step;
  double best_eff = -1.0;
  for (int j = 1; j <= jmax; ++j) {
    const int chunk = step * j;
    const long nwg = wgroups * ((K + chunk - 1) / chunk);
    const long rounds = (nwg + cus - 1) / cus;
    const double eff = (double)wgroups * K / ((double)rounds * cus * chunk);
    if (eff > best_eff + 1e-9 || (eff > best_eff - 1e-9 && chunk > best)) {
      best_eff = eff;
      best = chunk;
    }
  }
  return best;
}

}  // namespace

int exchange_i8w_chunks(int W, int N, int K) {
  const int chunk = chunk_of(W, N, K);
  return ((K + chunk - 1) / chunk) * (N > 16 ? 2 : 1);
}

void launch_exchange_i8w(hipStream_t s, int W, int M, int N, int K, const double* G, bool real,
                         const int8_t* Lq, const double* Lu, const int* ord, double* Kl, double* exx_part) {
  const int Mp = exchange_i8_row(M), chunk = chunk_of(W, N, K), nchunk = (K + chunk - 1) / chunk;
  const int wpb = N > 16 ? kT2Walkers : kWPB;
  const dim3 grid((W + wpb - 1) / wpb, nchunk), block(N > 16 ? 128 * kT2Walkers : 64 * kWPB);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, block, 0, s, W, M, N, K, Mp, chunk, G, Lq, Lu, ord, Kl, exx_part,
                       N > 16 ? 2 * nchunk : nchunk);
  };
  if (N > 16) {
    AFQ_CHECK(!real && M > 64, AFQ_EUNSUPPORTED, "int8 exchange per walker: 17 to 32 electrons need a complex "
              "trial on more than 64 orbitals");
    go(k_exchange_i8_w2);
  } else {
    if (real) M <= 64 ? go(k_exchange_i8_w1<1, 2, false>) : go(k_exchange_i8_w1<2, 1, false>);
    else M <= 64 ? go(k_exchange_i8_w1<1, 1, true>) : go(k_exchange_i8_w1<2, 1, true>);
  }
  AFQ_HIP(hipGetLastError());
}

}  // namespace afq
