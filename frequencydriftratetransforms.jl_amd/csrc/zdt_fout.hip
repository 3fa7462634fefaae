// Fused output for power-of-two Nf in [2^16, 2^22] and Nt <= FOUT_MAX_NT,
// where the chirp-Z coefficients of a bin do not fit k2's registers (Nt > 16)
// or the rows do not fit its LDS (Nf > 2^20):
//   k1_input + k2_input   input!: the four-step r2c into Ft[t][k2][k1]
//   czt_fold_col          the chirp-Z per bin -> Yc[j][k2][k1]
//   k2_c2r / k2_c2r_wave  c2r pre-pass and inverse DFT_N1 -> B (as k2)
//   k3_output             as in the fused path (fast_output)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "zdt_fast_dev.h"
#include "zdt_fast_plan.h"
#include "zdt_kernels.h"

namespace zdt {

// ---------------------------------------------------------------- fused output for Nt > 16
//
// For power-of-two Nf with Nt up to FOUT_MAX_NT (more coefficients than k2
// keeps in registers) the
// chirp-Z runs per bin (czt_fold_col) and the output irfft reuses the
// second half of k2 and k3:
//   czt_fold_col     Ys[k, j] -> Yc[j][k2][k1] (k = k2 + N2 k1 < M), Ys[M, j] -> yM[j]
//   k2_c2r           per Hermitian column pair: c2r pre-pass, inverse DFT_N1
//                    over k1 (one wavefront per row) -> B, bin M/2 -> yhalf
//   k3_output        as in the fused path
// which moves the spectra through HBM twice instead of once per FFT pass.

struct CztColArgs {
  const c32* F;  // [Nt][N2][N1] (bin k2 + N2 k1 at [t][k2][k1]) then [Nt] bin M
  c32* Yc;       // [Nr][N2][N1]
  c32* yM;       // [Nr]
  int64_t M, Nf;
  int logN1, logN2;
  FoldRates r;
  int past;      // store Yc past the last-level cache
  double r0, dr;
  int wkind;
  const float* wcustom;
  float scale;
};

// The chirp-Z of every bin, folded (czt_fold.h), for the rates in mirrored
// pairs about the centre rate rc = r0 + (Nr-1) dr/2: rates j and Nr-1-j are
// the sums at z = e^{2 pi i k (r_j - rc)/Nf} and conj(z) over the coefficients
// c_t e^{2 pi i k t rc/Nf}.  NC adjacent lanes share a bin (1 up to 80 time
// steps); bins g = 0 .. M-1 in the order of F and Yc (g = k1 + N1 k2), so that
// a block's loads and stores are contiguous runs.  The
// rate pairs are split over blockIdx.y.  VALU-bound from about 40 time steps
// on: 235 operations per bin and pair of rates at 64 steps (28 of them FP64),
// where the Reinsch recurrence it replaced took 395 and serialized its input
// loads.  Three wavefronts per SIMD up to 64 steps.  Measured, before -> after:
// 2^20 x 60 x 481 985 -> 689 us, 2^22 x 64 x 257 2229 -> 1556, 2^20 x 80 x 257
// 1043 -> 480 (two lanes a bin -> one), 2^16 x 279 x 257 342 -> 171; below 40
// steps the writes of Yc bound it (2^20 x 32 x 257 329 -> 244 us, 5.0 TB/s).
template <int NB, int NC>
__global__ __launch_bounds__(256, NB <= 4 ? 3 : 2) void czt_fold_col(CztColArgs a) {
  constexpr int BPB = 256 / NC;  // bins per block
  const int q = threadIdx.x % NC;
  const int64_t g = static_cast<int64_t>(blockIdx.x) * BPB + threadIdx.x / NC;  // < M
  const int64_t k = (g >> a.logN1) + ((g & ((int64_t(1) << a.logN1) - 1)) << a.logN2);
  FoldBin b;
  b.dst = a.Yc;
  b.stride = a.M;
  b.F = a.F;
  b.fs = a.M;
  b.o = static_cast<unsigned>(g);
  b.kd = static_cast<double>(k);
  b.w = fast_window(a.wkind, a.wcustom, k, a.Nf) * a.scale;
  const int npair = (a.r.Nr + 1) / 2;
  const int jlo = group_first(npair, blockIdx.y, gridDim.y), jhi = group_first(npair, blockIdx.y + 1, gridDim.y);
  if constexpr (NB == 0)
    short_rates<false>(b, a.r, jlo, jhi, a.past != 0);
  else
    fold_rates<NB, NC>(b, a.r, q, 0, jlo, jhi, false, a.past != 0);
  // the Nyquist bin, a wavefront per rate over all blocks (a block of its own
  // would cost a whole round where the others fill the chip exactly)
  const int lane = threadIdx.x & 63, nw = 4 * gridDim.x * gridDim.y;
  for (int j = 4 * (blockIdx.y * gridDim.x + blockIdx.x) + (threadIdx.x >> 6); j < a.r.Nr; j += nw) {
    const double rev = 0.5 * a.r0 + 0.5 * a.dr * static_cast<double>(j);  // e^{i pi t r_j}
    c32 s = {0.0f, 0.0f};
    for (int t = lane; t < a.r.Nt; t += 64) s = cfma(s, a.F[a.M * a.r.Nt + t], cis_nh(static_cast<double>(t), rev));
#pragma unroll
    for (int x = 32; x > 0; x >>= 1) {
      s.x += __shfl_xor(s.x, x, 64);
      s.y += __shfl_xor(s.y, x, 64);
    }
    const float w = fast_window(a.wkind, a.wcustom, a.M, a.Nf) * a.scale;
    if (lane == 0) a.yM[j] = {s.x * w, s.y * w};
  }
}

struct K2cArgs {
  const c32* Yc;  // [Nr][N2][N1]
  const c32* yM;  // [Nr]
  c32* B;         // [Nr][N1/16][N2][16]
  c32* yhalf;     // [Nr]
  const c32* tw1;
  int Nr;
  int64_t M, Nf;
  float oscale;   // output scale / M
};

__device__ __forceinline__ c32 load_nt(const c32* p) {
  typedef float f2v __attribute__((ext_vector_type(2)));
  const f2v v = __builtin_nontemporal_load(reinterpret_cast<const f2v*>(p));
  return {v.x, v.y};
}

// the rate loop of k2_czt with the spectra read from Yc instead of evaluated
template <int N1, int N2, int ROWS>
__global__ __launch_bounds__(N1 < 512 ? N1 : 512, k2_waves_per_eu(N1)) void k2_c2r(K2cArgs a) {
  constexpr int T = N1 < 512 ? N1 : 512;
  static_assert(T == N1, "one Hermitian pair per thread");
  constexpr int P = N1 + N1 / 8;
  constexpr int HALF = N1 / 2;
  __shared__ c32 buf[ROWS * P];
  __shared__ c32 buf2[ROWS * P];
  __shared__ c32 twl[N1 + N1 / 8];  // W_N1^m at lsw(m)
  for (int i = threadIdx.x; i < N1; i += T) twl[lsw(i)] = a.tw1[i];
  __syncthreads();
  const int tid = threadIdx.x;
  const int p = blockIdx.x;
  const bool special = (p == 0);
  const int colA = special ? 0 : p;
  const int colB = special ? N2 / 2 : N2 - p;
  const HPair hp = hpair<N1, N2>(p, tid);
  const int rowA = hp.rowA, rowB = hp.rowB, k1A = hp.k1A, k1B = hp.k1B, cA = hp.cA, cB = hp.cB;
  const bool nyq = hp.nyq;
  const int64_t kA = cA + static_cast<int64_t>(N2) * k1A;
  const c32 WA = cis_rev(-static_cast<float>(kA) / static_cast<float>(a.Nf));
  const float h = 0.5f * a.oscale;
  if (special && blockIdx.y == 0) {
    for (int j = tid; j < a.Nr; j += T) {
      const c32 y = a.Yc[static_cast<int64_t>(j) * a.M + HALF];  // bin M/2: k2 = 0, k1 = N1/2
      a.yhalf[j] = {y.x * a.oscale, -y.y * a.oscale};
    }
  }
  const c32* srcA = a.Yc + static_cast<int64_t>(cA) * N1 + k1A;
  const c32* srcB = a.Yc + static_cast<int64_t>(cB) * N1 + (nyq ? 0 : k1B);
  constexpr int JG = ROWS / 2;
  constexpr int NW = T / 64;
  constexpr int RPW = ROWS / NW;
  static_assert(RPW * NW == ROWS && RPW * fft_max_nr<N1>() <= 64, "one butterfly per lane and pass");
  const int wv = tid >> 6, lane = tid & 63;
  c32* cur = buf;
  c32* nxt = buf2;
  // the next group's spectra are loaded right after this group's barrier, so
  // their latency overlaps the inverse DFT
  c32 ya[JG], yb[JG];
  auto load = [&](int j0n) {
    const int njn = min(JG, a.Nr - j0n);
#pragma unroll
    for (int jj = 0; jj < JG; ++jj) {
      if (jj < njn) {
        const int64_t off = static_cast<int64_t>(j0n + jj) * a.M;
        ya[jj] = load_nt(srcA + off);
        yb[jj] = nyq ? a.yM[j0n + jj] : load_nt(srcB + off);
      }
    }
  };
  const int ng = (a.Nr + JG - 1) / JG;
  const int jlo = group_first(ng, blockIdx.y, gridDim.y) * JG;
  const int jhi = min(a.Nr, group_first(ng, blockIdx.y + 1, gridDim.y) * JG);
  load(jlo);
  for (int j0 = jlo; j0 < jhi; j0 += JG) {
    const int nj = min(JG, a.Nr - j0);
#pragma unroll
    for (int jj = 0; jj < JG; ++jj) {
      if (jj < nj) {
        const c32 YA = {ya[jj].x * h, ya[jj].y * h}, YB = {yb[jj].x * h, yb[jj].y * h};
        if (nyq) {
          cur[(2 * jj + rowA) * P] = {YA.x + YB.x, YA.x - YB.x};
          cur[(2 * jj + rowA) * P + lsw(HALF)] = {0.0f, 0.0f};
        } else {
          const c32 E = {YA.x + YB.x, YA.y - YB.y};
          const c32 D = {YA.x - YB.x, YA.y + YB.y};
          const c32 O = cmulc(D, WA);
          cur[(2 * jj + rowA) * P + lsw(k1A)] = {E.x - O.y, E.y + O.x};
          cur[(2 * jj + rowB) * P + lsw(k1B)] = {E.x + O.y, -E.y + O.x};
        }
      }
    }
    __syncthreads();
    if (j0 + JG < jhi) load(j0 + JG);
    const int nrw = min(RPW, max(0, 2 * nj - wv * RPW));
    wave_fft<N1, true, 1, true>(cur + wv * RPW * P, P, nrw, twl, lane, [&](int f, int jx, auto& v) {
      constexpr int RL = sizeof(v) / sizeof(c32);
      const int row = wv * RPW + f;
      c32* dst = a.B + static_cast<int64_t>(j0 + (row >> 1)) * (N1 * N2) + ((row & 1) ? colB : colA) * 16;
#pragma unroll
      for (int r = 0; r < RL; ++r) {
        const int n1 = jx + r * (N1 / RL);
        dst[(n1 >> 4) * (N2 * 16) + (n1 & 15)] = v[r];
      }
    });
    c32* t = cur;
    cur = nxt;
    nxt = t;
  }
}


// In-place inverse/forward FFT of one row of N entries owned by one
// wavefront, N/(64 R) radix-R butterflies per lane and pass (rows of 2^10 and
// 2^11 entries, too long for wave_fft's one butterfly per lane).  A pass
// issues all of its reads before any of its writes, as in wave_pass; the last
// pass calls emit(j, v) for each butterfly j of the lane (elements
// j + r N/R) instead of writing back.  Twiddles: the table tw of W_N^m.
template <int N, bool INV, int NS = 1, typename Emit>
__device__ __forceinline__ void wave_fft_row(c32* x, const c32* __restrict__ tw, int lane, Emit&& emit) {
  constexpr int R = fft_radix<N, NS>();
  constexpr int NR = N / R;
  constexpr int BPL = NR / 64;
  constexpr int LOGN = ilog2c(N), LOGR = ilog2c(R), LOGNS = ilog2c(NS);
  static_assert(BPL * 64 == NR && NR % 8 == 0, "whole butterflies per lane");
  c32 v[BPL][R];
#pragma unroll
  for (int b = 0; b < BPL; ++b) {
    const c32* xr = x + lsw(lane + 64 * b);
#pragma unroll
    for (int r = 0; r < R; ++r) v[b][r] = xr[r * (NR + NR / 8)];
  }
#pragma unroll
  for (int b = 0; b < BPL; ++b) {
    if constexpr (NS > 1) {
      const int k = (lane + 64 * b) & (NS - 1);
#pragma unroll
      for (int r = 1; r < R; ++r) {
        const c32 w = tw[(r * k) << (LOGN - LOGNS - LOGR)];
        v[b][r] = INV ? cmulc(v[b][r], w) : cmul(v[b][r], w);
      }
    }
    dftd<INV, float, R>(v[b]);
  }
  if constexpr (NS * R < N) {
#pragma unroll
    for (int b = 0; b < BPL; ++b) {
      const int j = lane + 64 * b;
      const int k = j & (NS - 1);
      c32* yy = x + lsw(((j >> LOGNS) << (LOGNS + LOGR)) + k);
      if constexpr (NS == 1) {
#pragma unroll
        for (int r = 0; r < R; ++r) yy[r + (r >> 3)] = v[b][r];
      } else {
#pragma unroll
        for (int r = 0; r < R; ++r) yy[r * (NS + (NS >> 3))] = v[b][r];
      }
    }
    wave_sync();
    wave_fft_row<N, INV, NS * R>(x, tw, lane, emit);
  } else {
#pragma unroll
    for (int b = 0; b < BPL; ++b) emit(lane + 64 * b, v[b]);
  }
}

// Inverse DFT of one 2048-entry row owned by one wavefront, in place and
// with 32 row entries per lane but at most 16 live at a time (a Stockham row
// FFT keeps all 32 live, which does not fit beside k2_c2r's state).  Stage 1
// is a radix-16 Stockham pass from natural order (butterfly j reads entries
// j + 128 r) whose outputs go to the digit-reversed positions of an in-place
// decimation-in-time FFT (group g = j/16 + 8 (j mod 16), entries 16 g + r');
// stages 2 (radix 8, span 16) and 3 (radix 16, span 128) are in-place DIT
// butterflies on entries g L + k + r L', one butterfly at a time, and stage 3
// calls emit(k, v) with v[r] = output k + 128 r.  Rows are stored with the
// swizzle s2048 (bits 7-10 folded into bits 0-3), which keeps every stage's
// accesses within two-way bank conflicts; tw is the LDS table of W_2048^m.
__device__ __forceinline__ int s2048(int i) { return i ^ ((i >> 7) & 15); }

template <typename Emit>
__device__ __forceinline__ void wave_ifft_2048(c32* x, const c32* tw, int lane, Emit&& emit) {
  // opaque to the optimizer: keeps the ~100 lane-dependent LDS addresses from
  // being hoisted out of the caller's rate loop (where they would spill)
  asm volatile("" : "+v"(lane));
  {
    c32 v[2][16];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) v[b][r] = x[s2048(lane + 64 * b + 128 * r)];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      dftd<true, float, 16>(v[b]);
      const int j = lane + 64 * b;
      const int g = (j >> 4) + 8 * (j & 15);
#pragma unroll
      for (int r = 0; r < 16; ++r) x[s2048(16 * g + r)] = v[b][r];
    }
  }
  wave_sync();
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int bb = lane + 64 * b;
    const int base = (bb >> 4) * 128 + (bb & 15);
    const int k = bb & 15;
    c32 v[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = x[s2048(base + 16 * r)];
#pragma unroll
    for (int r = 1; r < 8; ++r) v[r] = cmulc(v[r], tw[16 * r * k]);  // W_128^{-r k}
    dftd<true, float, 8>(v);
#pragma unroll
    for (int r = 0; r < 8; ++r) x[s2048(base + 16 * r)] = v[r];
  }
  wave_sync();
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int k = lane + 64 * b;
    c32 v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = x[s2048(k + 128 * r)];
#pragma unroll
    for (int r = 1; r < 16; ++r) v[r] = cmulc(v[r], tw[r * k]);  // W_2048^{-r k}
    dftd<true, float, 16>(v);
    emit(k, v);
  }
}

// k2_c2r for N1 = 1024, 2048 (Nf = 2^21, 2^22): ROWS wavefronts, PP = N1/(64
// ROWS) pairs per thread, groups of ROWS/2 rates (one row per wavefront) in
// one LDS buffer; each wavefront runs the inverse DFT_N1 of its row in place
// (wave_fft_row) and stores it, so a group costs two barriers.  Blocks walk the
// units (rate group, column pair), all pairs of a group before the next group:
// at N1 = 1024 as many blocks as the CUs hold, so that the few groups of a
// last-level-cache chunk (see fast_out_run) keep every CU busy; at N1 = 2048
// (no chunks) a block per pair.  The next unit's spectra are loaded into registers before the DFTs,
// so their latency overlaps them.  At 2^22 x 257 it moves its 8.6 GB in 1.78 ms
// (4.8 TB/s, a copy's rate); ROWS = 4 with two blocks a CU took 2.28 ms there,
// but at N1 = 1024 four blocks of ROWS = 4 beat two of 8 (2^21 x 257 in
// chunks: 890 against 928 us).
template <int N1, int N2, int ROWS>
__global__ __launch_bounds__(64 * ROWS, 2) void k2_c2r_wave(K2cArgs a) {
  constexpr int T = 64 * ROWS;
  constexpr int PP = N1 / T;
  constexpr bool BIG = N1 == 2048;  // wave_ifft_2048 layout (no row padding)
  constexpr int P = BIG ? N1 : N1 + N1 / 8;
  constexpr int HALF = N1 / 2;
  constexpr int JG = ROWS / 2;
  __shared__ c32 buf[ROWS * P];
  __shared__ c32 twl[BIG ? N1 : 1];
  if constexpr (BIG) {
    for (int i = threadIdx.x; i < N1; i += T) twl[i] = a.tw1[i];
  }
  auto pos = [](int i) { return BIG ? s2048(i) : lsw(i); };
  const int tid = threadIdx.x;
  const float h = 0.5f * a.oscale;
  const float invNf = 1.0f / static_cast<float>(a.Nf);
  const int units = (a.Nr + JG - 1) / JG * (N2 / 2);
  c32 ya[JG][PP], yb[JG][PP];
  auto load = [&](int u) {
    const int p = u % (N2 / 2), j0 = u / (N2 / 2) * JG;
#pragma unroll
    for (int i = 0; i < PP; ++i) {
      const HPair q = hpair<N1, N2>(p, tid + i * T);
      const int oa = q.cA * N1 + q.k1A, ob = q.cB * N1 + (q.nyq ? 0 : q.k1B);
#pragma unroll
      for (int jj = 0; jj < JG; ++jj) {
        if (j0 + jj < a.Nr) {  // uniform
          const c32* y = a.Yc + static_cast<int64_t>(j0 + jj) * a.M;  // uniform
          ya[jj][i] = load_nt(y + oa);
          yb[jj][i] = q.nyq ? a.yM[j0 + jj] : load_nt(y + ob);
        }
      }
    }
  };
  int u = blockIdx.x;
  if (u < units) load(u);
  const int wv = tid >> 6, lane = tid & 63;
  for (; u < units; u += gridDim.x) {
    const int p = u % (N2 / 2), j0 = u / (N2 / 2) * JG;
    const int nj = min(JG, a.Nr - j0);
#pragma unroll
    for (int i = 0; i < PP; ++i) {
      const HPair q = hpair<N1, N2>(p, tid + i * T);
      const c32 WA = cis_rev(-static_cast<float>(q.cA + N2 * q.k1A) * invNf);
#pragma unroll
      for (int jj = 0; jj < JG; ++jj) {
        if (jj < nj) {
          const c32 YA = {ya[jj][i].x * h, ya[jj][i].y * h}, YB = {yb[jj][i].x * h, yb[jj][i].y * h};
          if (q.nyq) {
            buf[(2 * jj + q.rowA) * P] = {YA.x + YB.x, YA.x - YB.x};
            buf[(2 * jj + q.rowA) * P + pos(HALF)] = {0.0f, 0.0f};
          } else {
            const c32 E = {YA.x + YB.x, YA.y - YB.y};
            const c32 D = {YA.x - YB.x, YA.y + YB.y};
            const c32 O = cmulc(D, WA);
            buf[(2 * jj + q.rowA) * P + pos(q.k1A)] = {E.x - O.y, E.y + O.x};
            buf[(2 * jj + q.rowB) * P + pos(q.k1B)] = {E.x + O.y, -E.y + O.x};
          }
        }
      }
    }
    if (p == 0 && tid < nj) {  // the bin M/2: k2 = 0, k1 = N1/2
      const c32 y = a.Yc[static_cast<int64_t>(j0 + tid) * a.M + HALF];
      a.yhalf[j0 + tid] = {y.x * a.oscale, -y.y * a.oscale};
    }
    __syncthreads();
    if (u + static_cast<int>(gridDim.x) < units) load(u + gridDim.x);
    if (wv < 2 * nj) {  // uniform per wavefront: wavefront wv owns row wv
      const int col = p == 0 ? (wv & 1) * (N2 / 2) : ((wv & 1) ? N2 - p : p);
      c32* dst = a.B + static_cast<int64_t>(j0 + (wv >> 1)) * (N1 * N2) + col * 16;
      auto emit = [&](int jx, auto& v) {
        constexpr int RL = sizeof(v) / sizeof(c32);
#pragma unroll
        for (int r = 0; r < RL; ++r) {
          const int n1 = jx + r * (N1 / RL);
          dst[(n1 >> 4) * (N2 * 16) + (n1 & 15)] = v[r];
        }
      };
      if constexpr (BIG) {
        wave_ifft_2048(buf + wv * P, twl, lane, emit);
      } else {
        int ln = lane;
        asm volatile("" : "+v"(ln));  // keeps the row FFT's LDS addresses inside the rate loop
        wave_fft_row<N1, true>(buf + wv * P, a.tw1, ln, emit);
      }
    }
    __syncthreads();  // the rows are rewritten by the next unit
  }
}

// ---------------------------------------------------------------- fused-output input

struct K2iArgs {
  c32* G;          // in: [Nt][N2][N1] column FFTs of k1_input; out: X_t(k2 + N2 k1) at [t][k2][k1]
  c32* XM;         // [Nt] X_t(M)
  const c32* tw1;  // W_N1^m
  int Nt;
  int64_t M, Nf;
};

// input! for the fused output: the second half of the four-step r2c, in
// place over k1_input's G.  Block per Hermitian column pair as in k2_czt
// (regular block p: columns p and N2-p; block 0: columns 0 and N2/2); for each
// group of TG = ROWS/2 time steps the 2 TG rows get the twiddle W_M^{n1 k2}
// and a forward DFT_N1, then each thread untangles its pairs (k, M-k) into
// the r2c spectrum and writes both bins back over the rows it read.  Bound by
// HBM now (4.4 TB/s for its read and write of G at 2^22 x 64): loading the next
// group's rows before the DFT and the twiddle table from LDS instead of
// global memory took 2^22 x 64 from 772 to 491 us, 2^21 x 32 from 210 to 127 and
// 2^20 x 60 from 165 to 110.
template <int N1, int N2, int ROWS>
__global__ __launch_bounds__(N1 < 1024 ? N1 : 1024) void k2_input(K2iArgs a) {
  constexpr int T = N1 < 1024 ? N1 : 1024;
  constexpr int PP = N1 / T;
  constexpr int P = N1 + N1 / 8;
  constexpr int HALF = N1 / 2;
  constexpr int TG = ROWS / 2;
  __shared__ c32 buf[ROWS * P];
  __shared__ c32 buf2[ROWS * P];
  __shared__ c32 twl[N1 + N1 / 8];  // W_N1^m at lsw(m)
  for (int i = threadIdx.x; i < N1; i += T) twl[lsw(i)] = a.tw1[i];
  const int tid = threadIdx.x;
  const int p = blockIdx.x;
  const bool special = (p == 0);
  const int colA = special ? 0 : p;
  const int colB = special ? N2 / 2 : N2 - p;

  int rowA[PP], rowB[PP], k1A[PP], k1B[PP];
  bool nyq[PP];
  c32 WA[PP], twS0[PP], twS1[PP];
  const float invM = 1.0f / static_cast<float>(a.M);
#pragma unroll
  for (int i = 0; i < PP; ++i) {
    const int q = tid + i * T;
    const HPair h = hpair<N1, N2>(p, q);
    rowA[i] = h.rowA;
    rowB[i] = h.rowB;
    k1A[i] = h.k1A;
    k1B[i] = h.k1B;
    nyq[i] = h.nyq;
    const int cA = h.cA;
    const int64_t kA = cA + static_cast<int64_t>(N2) * k1A[i];
    WA[i] = cis_rev(-static_cast<float>(kA) / static_cast<float>(a.Nf));  // W_Nf^{kA}
    const int64_t n1 = q;
    twS0[i] = cis_rev(static_cast<float>((n1 * colA) & (a.M - 1)) * invM);
    twS1[i] = cis_rev(static_cast<float>((n1 * colB) & (a.M - 1)) * invM);
  }

  const int ng = (a.Nt + TG - 1) / TG;
  const int tlo = group_first(ng, blockIdx.y, gridDim.y) * TG;
  const int thi = min(a.Nt, group_first(ng, blockIdx.y + 1, gridDim.y) * TG);
  // the next group's rows are loaded before this group's DFT
  c32 v[ROWS][PP];
  auto load = [&](int t0) {
    const int nt = min(TG, a.Nt - t0);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      if (r < 2 * nt) {
        const c32* src = a.G + (static_cast<int64_t>(t0 + (r >> 1)) * N2 + ((r & 1) ? colB : colA)) * N1;
#pragma unroll
        for (int i = 0; i < PP; ++i) v[r][i] = src[tid + i * T];
      }
    }
  };
  load(tlo);
  for (int t0 = tlo; t0 < thi; t0 += TG) {
    const int nt = min(TG, a.Nt - t0);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      if (r < 2 * nt) {
#pragma unroll
        for (int i = 0; i < PP; ++i)
          buf[r * P + lsw(tid + i * T)] = cmulc(v[r][i], (r & 1) ? twS1[i] : twS0[i]);
      }
    }
    if (t0 + TG < thi) load(t0 + TG);
    __syncthreads();
    const c32* fz = lds_fft_pp<N1, T, false, 1, true>(buf, buf2, P, 2 * nt, twl);
#pragma unroll
    for (int uu = 0; uu < TG; ++uu) {
      if (uu < nt) {
        const int64_t t = t0 + uu;
        c32* rA = a.G + (t * N2 + colA) * N1;
        c32* rB = a.G + (t * N2 + colB) * N1;
#pragma unroll
        for (int i = 0; i < PP; ++i) {
          const c32 Za = fz[(2 * uu + rowA[i]) * P + lsw(k1A[i])];
          c32* dA = rowA[i] ? rB : rA;
          c32* dB = rowB[i] ? rB : rA;
          if (nyq[i]) {
            dA[0] = {Za.x + Za.y, 0.0f};
            a.XM[t] = {Za.x - Za.y, 0.0f};
          } else {
            const c32 Zb = fz[(2 * uu + rowB[i]) * P + lsw(k1B[i])];
            const c32 E = {0.5f * (Za.x + Zb.x), 0.5f * (Za.y - Zb.y)};
            const c32 O = {0.5f * (Za.y + Zb.y), -0.5f * (Za.x - Zb.x)};
            const c32 WO = cmul(WA[i], O);
            dA[k1A[i]] = cadd(E, WO);
            dB[k1B[i]] = {E.x - WO.x, -(E.y - WO.y)};
          }
        }
        if (special && tid == 0) {
          // bin M/2 (column 0, k1 = N1/2) is its own partner: X = conj(Z)
          const c32 Zh = fz[(2 * uu) * P + lsw(HALF)];
          rA[HALF] = cconj(Zh);
        }
      }
    }
    __syncthreads();
  }
}

// F (natural Nk x Nt) from the fused-output input layout
__global__ __launch_bounds__(256) void ft_to_natural(const c32* __restrict__ Ft, c32* __restrict__ F, int64_t Nk,
                                                     int Nt, int logN1, int logN2) {
  const int64_t M = Nk - 1;
  const int64_t total = Nk * Nt;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < total;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t t = g / Nk, k = g - t * Nk;
    const int64_t k2 = k & ((int64_t(1) << logN2) - 1), k1 = k >> logN2;
    F[g] = (k == M) ? Ft[M * Nt + t] : Ft[t * M + (k2 << logN1) + k1];
  }
}

}  // namespace zdt

namespace zdt {

// ---------------------------------------------------------------- fused output (host)

// bytes of spectra per chunk of rates (see fast_out_run)
constexpr int64_t FOUT_CHUNK = int64_t(224) << 20;

bool fast_out_supported(int64_t Nf, int64_t Nt, int64_t Nr) {
  if (Nf < (1 << 16) || Nf > (1 << 22) || (Nf & (Nf - 1)) != 0) return false;
  return Nt >= 1 && Nt <= FOUT_MAX_NT && Nr >= 1 && Nr <= 65535;
}

int64_t fast_out_bytes(int64_t Nf, int64_t Nr) {
  const int64_t M = Nf / 2;
  const int64_t N2 = fast_n2(Nf);
  return 16 * M * Nr + 8 * (M / N2 + N2 + 2 * Nr) + 8 * fast_stats_doubles(Nf, Nr);
}

int fast_out_create(int64_t Nf, int64_t Nr, int precision, FastPlan** out) {
  *out = nullptr;
  if (!fast_out_supported(Nf, 1, Nr)) return fail(ZDT_ENOTSUP, "fused output: unsupported shape");
  if (!fast_precision_ok(Nf, 0, precision))
    return fail(ZDT_ENOTSUP, "fused output: precision %d not available for Nf=%lld", precision, (long long)Nf);
  FastPlan* p = new FastPlan();
  p->precision = precision;
  p->Nf = Nf;
  p->Nt = 0;
  p->Nr = Nr;
  p->M = Nf / 2;
  p->N2 = fast_n2(Nf);
  p->logN2 = ilog2i(p->N2);
  p->N1 = static_cast<int>(p->M / p->N2);
  p->logN1 = ilog2i(p->N1);
  {
    int dev = 0, ncu = 256;
    if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    p->resident_blocks = 2 * static_cast<int64_t>(ncu);
  }
  int rc = ZDT_OK;
  auto alloc = [&](c32** q, size_t n) {
    if (rc != ZDT_OK) return;
    hipError_t e = hipMalloc(reinterpret_cast<void**>(q), n * sizeof(c32));
    if (e != hipSuccess) {
      (void)hipGetLastError();
      rc = fail(ZDT_ENOMEM, "hipMalloc(%zu bytes) failed: %s", n * sizeof(c32), hipGetErrorString(e));
    }
  };
  alloc(&p->Yc, static_cast<size_t>(Nr * p->M));
  alloc(&p->B, static_cast<size_t>(Nr * p->M));
  alloc_part(p, rc);
  alloc(&p->yM, static_cast<size_t>(Nr));
  alloc(&p->yhalf, static_cast<size_t>(Nr));
  if (rc == ZDT_OK) rc = upload_table(&p->tw1, twiddles(p->N1));
  if (rc == ZDT_OK) rc = upload_table(&p->tw2, twiddles(p->N2));
  if (rc != ZDT_OK) {
    fast_destroy(p);
    return rc;
  }
  *out = p;
  return ZDT_OK;
}

template <int N1, int N2>
static int launch_k2c(const K2cArgs& a, int64_t ncu, hipStream_t st) {
  if constexpr (N1 <= 512) {
    // rate groups over blockIdx.y: at 257 rates, one part -> this rule, 2^16
    // channels 79.6 -> 24.0 us, 2^17 86.8 -> 51, 2^18 123 -> 100, 2^19
    // 227 -> 220; nothing at 2^20
    constexpr int JG = k2_rows(N1) / 2;
    const dim3 grid(N2 / 2, group_parts((a.Nr + JG - 1) / JG, N2 / 2, N1, 24, 2, ncu));
    k2_c2r<N1, N2, k2_rows(N1)><<<grid, N1, 0, st>>>(a);
  } else {
    constexpr int ROWS = N1 == 2048 ? 8 : 4;
    const int64_t units = static_cast<int64_t>((a.Nr + ROWS / 2 - 1) / (ROWS / 2)) * (N2 / 2);
    const unsigned grid = static_cast<unsigned>(std::min<int64_t>(units, N1 == 2048 ? N2 / 2 : 4 * ncu));
    k2_c2r_wave<N1, N2, ROWS><<<grid, 64 * ROWS, 0, st>>>(a);
  }
  ZDT_CHECK_LAUNCH("k2_c2r");
  return ZDT_OK;
}

template <int N1, int N2>
static void launch_k2i(const K2iArgs& a, int64_t ncu, hipStream_t st) {
  // two ping-pong buffers of ~36 KB each: 8 rows up to N1 = 512, then 4, 2
  constexpr int ROWS = N1 <= 512 ? 8 : (N1 == 1024 ? 4 : 2);
  // groups of time steps over blockIdx.y up to 16 wavefronts a CU (the LDS
  // rows bound them there from N1 = 512 on): 2^16 x 279 247 -> 33 us, 2^17 x
  // 60 57.9 -> 20, 2^18 x 60 64.5 -> 28.9, 2^19 x 32 45.1 -> 32.4
  constexpr int T = N1 < 1024 ? N1 : 1024;
  const dim3 grid(N2 / 2, group_parts((a.Nt + ROWS / 2 - 1) / (ROWS / 2), N2 / 2, T, 16, 1, ncu));
  k2_input<N1, N2, ROWS><<<grid, T, 0, st>>>(a);
}

int fast_out_input(FastPlan* p, const float* spec, int64_t Nt, c32* Ft, hipStream_t st) {
  if (Nt < 1 || Nt > FOUT_MAX_NT) return fail(ZDT_ENOTSUP, "fused output: Nt=%lld", (long long)Nt);
  ZDT_TRY(launch_k1(p, spec, Ft, Nt, st));
  K2iArgs a;
  a.G = Ft;
  a.XM = Ft + p->M * Nt;
  a.tw1 = p->tw1;
  a.Nt = static_cast<int>(Nt);
  a.M = p->M;
  a.Nf = p->Nf;
  ProfScope ps(st, "k2_input", 16.0 * p->M * Nt);
  switch (p->N1 * 2048 + p->N2) {
    case 64 * 2048 + 512:
      launch_k2i<64, 512>(a, p->resident_blocks / 2, st);
      break;
    case 64 * 2048 + 1024:
      launch_k2i<64, 1024>(a, p->resident_blocks / 2, st);
      break;
    case 128 * 2048 + 1024:
      launch_k2i<128, 1024>(a, p->resident_blocks / 2, st);
      break;
    case 256 * 2048 + 1024:
      launch_k2i<256, 1024>(a, p->resident_blocks / 2, st);
      break;
    case 512 * 2048 + 1024:
      launch_k2i<512, 1024>(a, p->resident_blocks / 2, st);
      break;
    case 1024 * 2048 + 1024:
      launch_k2i<1024, 1024>(a, p->resident_blocks / 2, st);
      break;
    case 2048 * 2048 + 1024:
      launch_k2i<2048, 1024>(a, p->resident_blocks / 2, st);
      break;
    default:
      return fail(ZDT_ENOTSUP, "fused output input: N1=%d N2=%d", p->N1, p->N2);
  }
  ZDT_CHECK_LAUNCH("k2_input");
  return ZDT_OK;
}

int fast_out_unpack_F(FastPlan* p, const c32* Ft, int64_t Nt, c32* F, hipStream_t st) {
  const int64_t n = (p->M + 1) * Nt;
  int64_t g = (n + 255) / 256;
  if (g > (1 << 20)) g = 1 << 20;
  ft_to_natural<<<static_cast<unsigned>(g), 256, 0, st>>>(Ft, F, p->M + 1, static_cast<int>(Nt), p->logN1, p->logN2);
  ZDT_CHECK_LAUNCH("ft_to_natural");
  return ZDT_OK;
}

static int run_k2c(const FastPlan* p, const K2cArgs& a, hipStream_t st) {
  ProfScope ps(st, "k2_c2r", 16.0 * p->M * a.Nr);
  switch (p->N1 * 2048 + p->N2) {
    case 64 * 2048 + 512:
      ZDT_TRY((launch_k2c<64, 512>(a, p->resident_blocks / 2, st)));
      break;
    case 64 * 2048 + 1024:
      ZDT_TRY((launch_k2c<64, 1024>(a, p->resident_blocks / 2, st)));
      break;
    case 128 * 2048 + 1024:
      ZDT_TRY((launch_k2c<128, 1024>(a, p->resident_blocks / 2, st)));
      break;
    case 256 * 2048 + 1024:
      ZDT_TRY((launch_k2c<256, 1024>(a, p->resident_blocks / 2, st)));
      break;
    case 512 * 2048 + 1024:
      ZDT_TRY((launch_k2c<512, 1024>(a, p->resident_blocks / 2, st)));
      break;
    case 1024 * 2048 + 1024:
      ZDT_TRY((launch_k2c<1024, 1024>(a, p->resident_blocks / 2, st)));
      break;
    case 2048 * 2048 + 1024:
      ZDT_TRY((launch_k2c<2048, 1024>(a, p->resident_blocks / 2, st)));
      break;
    default:
      return fail(ZDT_ENOTSUP, "fused output: N1=%d N2=%d", p->N1, p->N2);
  }
  return ZDT_OK;
}

int fast_out_run(FastPlan* p, const c32* F, int Nt, float r0, float dr, int wkind, const float* window, float* dest,
                 double scale, hipStream_t st, double* colmean, double* colvar) {
  if (Nt < 1 || Nt > FOUT_MAX_NT) return fail(ZDT_ENOTSUP, "fused output: Nt=%d", Nt);
  // Rates in chunks whose spectra B (written by k2_c2r, read once by k3) stay
  // in the 256 MB last-level cache: every chunk reuses the start of p->B, Yc is
  // read and the FDR written past the cache (nontemporal).  A copy from there
  // runs at 7-8 TB/s against 5.5 from HBM.  224 MB a chunk: smaller ones pay
  // more launches and tails, larger ones spill (2^20 x 60 x 481, whole call:
  // 2555 us in one piece, 2457, 2412, 2395, 2358 in chunks of 128, 160, 192, 224
  // MB).  Not at 2^22, whose k2_c2r_wave has one block a CU and loses what k3
  // gains (6090 and 6155 us).  Without dest, p->B holds every rate for output!.
  const int64_t rate_bytes = 8 * p->M;
  int64_t per = p->Nr;
  if (dest != nullptr && p->N1 <= 1024 && rate_bytes * p->Nr > FOUT_CHUNK + FOUT_CHUNK / 8) {
    const int64_t nch = (rate_bytes * p->Nr + FOUT_CHUNK - 1) / FOUT_CHUNK;
    const int64_t r = p->N1 <= 512 ? 8 : 4;  // whole rate groups and, at 2^20, whole rounds of k3's tiles
    per = ((p->Nr + nch - 1) / nch + r - 1) / r * r;
  }
  const bool chunked = per < p->Nr;
  CztColArgs c;
  c.F = F;
  c.Yc = p->Yc;
  c.yM = p->yM;
  c.M = p->M;
  c.Nf = p->Nf;
  c.logN1 = p->logN1;
  c.logN2 = p->logN2;
  c.r0 = static_cast<double>(r0);
  c.dr = static_cast<double>(dr);
  c.wkind = wkind;
  c.wcustom = window;
  c.scale = 1.0f;
  // rates in mirrored pairs around the centre rate (a single rate is its own partner)
  const double rc = static_cast<double>(r0) + 0.5 * static_cast<double>(p->Nr - 1) * static_cast<double>(dr);
  const double nf = static_cast<double>(p->Nf);
  c.r = {Nt, static_cast<int>(p->Nr), static_cast<double>(dr) / nf, rc / nf, (static_cast<double>(r0) - rc) / nf};
  {
    int nb = 0, nc = 0;
    fold_split(Nt, 0, &nb, &nc);
    // (Yc in rate chunks is read past the cache too: see below)
    c.past = fold_past(8 * p->M * p->Nr, nb) || chunked ? 1 : 0;
    const int bpb = 256 / nc;  // bins per block
    const int nblk = static_cast<int>(p->M / bpb);
    // rate pairs over blockIdx.y up to the wavefronts a CU holds (8 with five
    // blocks of coefficients, 12 with fewer); a part repeats the coefficients,
    // worth about ten pairs
    const dim3 grid(static_cast<unsigned>(nblk), group_parts(static_cast<int>((p->Nr + 1) / 2), nblk, 256,
                                                             nb == 5 ? 8 : 12, 24, p->resident_blocks / 2));
    ProfScope ps(st, "czt_fold_col", 8.0 * (p->M + 1) * (Nt + p->Nr));  // F read, Yc written, once each
    if (!fold_dispatch(nb, nc, [&](auto B, auto C) { czt_fold_col<B(), C()><<<grid, 256, 0, st>>>(c); }))
      return fail(ZDT_ENOTSUP, "fused output: Nt=%d", Nt);
    ZDT_CHECK_LAUNCH("czt_fold_col");
  }
  K2cArgs a;
  a.B = p->B;
  a.tw1 = p->tw1;
  a.M = p->M;
  a.Nf = p->Nf;
  a.oscale = static_cast<float>(scale / static_cast<double>(p->M));
  for (int64_t j0 = 0; j0 < p->Nr; j0 += per) {
    const int64_t n = std::min(per, p->Nr - j0);
    a.Yc = p->Yc + j0 * p->M;
    a.yM = p->yM + j0;
    a.yhalf = p->yhalf + j0;
    a.Nr = static_cast<int>(n);
    ZDT_TRY(run_k2c(p, a, st));
    if (dest != nullptr) ZDT_TRY(fast_output_part(p, dest, j0, n, st, colmean != nullptr));
  }
  p->have_B = per >= p->Nr;
  if (colmean != nullptr && dest != nullptr) ZDT_TRY(fast_stats_merge(p, st, colmean, colvar));
  return ZDT_OK;
}

// Each piece reads F again: 64 rates of 16 steps in one piece take 1171 us where
// 14 at a time take 1387 (2^22), 595 against 640 (2^21), and 128 rates 572 against 551
// (2^20).  Above 2^20 the bound is for the memory kept, 470 MB.
int64_t fast_rates_chunk(int64_t Nf) { return std::max<int64_t>(1, FOUT_CHUNK / (4 * Nf)); }

size_t fast_rates_bytes(int64_t Nf, int64_t n) { return static_cast<size_t>(n * (Nf + 2)) * sizeof(c32); }

int fast_out_rates(const FastPlan* p, void* buf, int64_t n, const c32* F, int Nt, const double* rates_over_nf,
                   int64_t Nr, float* dest, hipStream_t st) {
  // p's shape and tables, buf's spectra
  FastPlan q = *p;
  q.precision = ZDT_PRECISION_FP32;
  q.paired = false;
  q.smax = nullptr;
  q.Yc = static_cast<c32*>(buf);
  q.B = q.Yc + n * q.M;
  q.yM = q.B + n * q.M;
  q.yhalf = q.yM + n;
  // pieces whose spectra B stay in the last-level cache, as in fast_out_run
  for (int64_t j0 = 0; j0 < Nr; j0 += n) {
    const int64_t m = std::min(n, Nr - j0);
    CztRatesArgs c;
    c.F = F;
    c.fs = q.M;
    c.Ys = q.Yc;
    c.ys = q.M;
    c.n = q.M;
    c.logN1 = q.logN1;
    c.logN2 = q.logN2;
    c.yM = q.yM;
    c.Nt = Nt;
    ZDT_TRY(launch_czt_rates(c, rates_over_nf + j0, m, st));
    K2cArgs a;
    a.Yc = q.Yc;
    a.yM = q.yM;
    a.B = q.B;
    a.yhalf = q.yhalf;
    a.tw1 = q.tw1;
    a.Nr = static_cast<int>(m);
    a.M = q.M;
    a.Nf = q.Nf;
    a.oscale = static_cast<float>(1.0 / static_cast<double>(q.M));
    ZDT_TRY(run_k2c(&q, a, st));
    ZDT_TRY(fast_output_part(&q, dest + j0 * q.Nf, 0, m, st, false));
  }
  return ZDT_OK;
}

}  // namespace zdt
