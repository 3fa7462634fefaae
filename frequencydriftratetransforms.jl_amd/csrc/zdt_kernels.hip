// ZDT kernels of the generic path and the step functions.
//
// The chirp-Z transform per frequency bin k (src/zdtfdr.jl:196-321) is
//   Ys[k,j] = post(k,j) w(k) sum_t F[k,t] pre(k,t) chirp(k, j-t),   j < Nr
// with chirp(k,l) = exp(-i pi k l^2 dr/Nf)                       (:140-142)
//      pre(k,t)   = exp( i pi k t (t dr + 2 r0)/Nf)              (:196-198)
//      post(k,j)  = exp( i pi k j^2 dr/Nf) = conj(chirp(k,j))    (:268-270)
// The reference evaluates the convolution over t as a length-Nl circular
// convolution through FFTs (:249-253); the identity chirp(k,l) = chirp(k,-l)
// makes the high lags of V (:182-184) the negative lags, so the result equals
// the linear convolution above for any Nl >= Nt+Nr-1.  czt_fold evaluates it
// directly (two to three operations per time step and output), which costs
// less than the two length-Nl FFTs, needs no V, and is exact up to float
// rounding.  The step functions (preprocess!,
// convolve!, postprocess!) keep the reference's FFT data flow on the
// materialized Nk x Nl matrix Y for API parity.
#include <hip/hip_runtime.h>

#include "czt_fold.h"
#include "zdt_fast_plan.h"
#include "zdt_kernels.h"

namespace zdt {

// exp(2 pi i rev) in double for any rev (reduced first)
__device__ __forceinline__ c64 cis64(double rev) {
  const double f = rev - __builtin_rint(rev);
  double s, c;
  sincospi(2.0 * f, &s, &c);
  return {c, s};
}

// exp(2 pi i (n1*h1 + n2*h2)) in float, each product reduced mod 1 in double
__device__ __forceinline__ c32 cis_sum2(double n1, double h1, double n2, double h2) {
  double p1 = n1 * h1;
  p1 -= __builtin_rint(p1);
  double p2 = n2 * h2;
  p2 -= __builtin_rint(p2);
  double p = p1 + p2;
  p -= __builtin_rint(p);
  return cis_rev(static_cast<float>(p));
}

__device__ __forceinline__ float window_value(int wkind, const float* wcustom, int64_t k, int64_t Nf) {
  if (wkind == ZDT_WINDOW_HAMMING) {
    // 0.53836 + 0.46164 cospi(2k/Nf)  (src/zdtfdr.jl:303-305)
    double p = static_cast<double>(k) / static_cast<double>(Nf);
    p -= __builtin_rint(p);
    const c32 c = cis_rev(static_cast<float>(p));
    return 0.53836f + 0.46164f * c.x;
  }
  if (wkind == ZDT_WINDOW_CUSTOM) return wcustom[k];
  return 1.0f;
}

// ---------------------------------------------------------------------------
// The chirp-Z of every bin (natural layout): by Bluestein's identity the sum
// above is Ys[k,j] = w(k) sum_t a_t z_j^t, a_t = F[k,t] e^{2 pi i k t r0/Nf},
// z_j = e^{2 pi i k j dr/Nf}, taken for mirrored pairs of rates about the
// centre rate by the fold of czt_fold.h, NC lanes per bin.  The rate pairs are
// split over blockIdx.y; sums longer than FOLD_MAX_NT take one launch per
// FOLD_MAX_NT steps, the later ones (tbase > 0) adding to Ys.  Bound by the
// writes of Ys from about 10^5 bins on (10^6 channels x 16 x 129: 128 -> 111 us,
// 5.2 TB/s, with Ys in columns of whole cache lines), below by latency: all input loads are in flight together, where the Reinsch
// kernels this replaced waited for each and reread Ys for every 64 steps past
// the first (4096 x 16 x 33 11.2 -> 7.5 us, 4096 x 60 x 257 130 -> 23, 2^15 x 177 x
// 394 611 -> 118, 21609 x 234 x 205 465 -> 66).
//
// Odd Nf, whose c2r takes two rates a transform: *a.wide tells that values come
// near overflow or are not finite, so that the c2r keeps the rates apart;
// the flag of the run after this one is cleared.
template <int NB, int NC>
__global__ __launch_bounds__(256, NB <= 4 ? 3 : 2) void czt_fold(CztArgs a, int tbase, int past) {
  constexpr int BPB = 256 / NC;  // bins per block
  const int64_t k = static_cast<int64_t>(blockIdx.x) * BPB + threadIdx.x / NC;
  if (k >= a.Nk) return;  // whole groups of NC lanes leave together
  FoldBin b;
  b.F = a.F;
  b.fs = a.ldF;
  b.dst = a.Ys;
  b.stride = a.ldY;
  b.o = static_cast<unsigned>(k);
  b.kd = static_cast<double>(k);
  b.w = window_value(a.wkind, a.wcustom, k, a.Nf) * a.scale;
  b.wide = a.wide;
  const FoldRates r = {a.Nt, a.Nr, 2.0 * a.hd, a.hc, a.hz};
  const int npair = (a.Nr + 1) / 2;
  const int jlo = group_first(npair, blockIdx.y, gridDim.y), jhi = group_first(npair, blockIdx.y + 1, gridDim.y);
  if constexpr (NB == 0)
    short_rates<true>(b, r, jlo, jhi, past != 0);
  else
    fold_rates<NB, NC, true>(b, r, threadIdx.x % NC, tbase, jlo, jhi, tbase > 0, past != 0);
  if (a.wide != nullptr && k == 0 && blockIdx.y == 0 && threadIdx.x == 0)
    *reinterpret_cast<int*>(reinterpret_cast<uintptr_t>(a.wide) ^ 4) = 0;
}

int launch_czt(const CztArgs& a, hipStream_t st) {
  int dev = 0, ncu = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  ProfScope ps(st, "czt_fold", 8.0 * static_cast<double>(a.Nk) * (a.Nt + a.Nr));
  for (int tbase = 0; tbase < a.Nt; tbase += FOLD_MAX_NT) {
    int nb = 0, nc = 0;
    fold_split(a.Nt, tbase, &nb, &nc);
    const int per = 256 / nc;
    const int nblk = static_cast<int>((a.Nk + per - 1) / per);
    // (whole cache lines: a 128-byte aligned destination and column stride)
    const int past = fold_past(8 * a.Nk * a.Nr, nb) && a.ldY % 16 == 0 ? 1 : 0;
    // rate pairs over blockIdx.y up to the wavefronts a CU holds; a part repeats
    // the coefficients
    const dim3 grid(static_cast<unsigned>(nblk),
                    group_parts((a.Nr + 1) / 2, nblk, 256, nb == 5 ? 8 : 12, 4 * (nb + 1), ncu));
    if (!fold_dispatch(nb, nc, [&](auto B, auto C) { czt_fold<B(), C()><<<grid, 256, 0, st>>>(a, tbase, past); }))
      return fail(ZDT_ENOTSUP, "chirp-Z: Nt=%d", a.Nt);
    ZDT_CHECK_LAUNCH("czt_fold");
  }
  return ZDT_OK;
}

// ---------------------------------------------------------------------------
// fftfdr (src/fftfdr.jl:86-96,126-148) for an arbitrary list of rates:
//   Ys[k,j] = sum_t F[k,t] e^{2 pi i k t rates[j]/Nf}.
// Per bin and rate z = e^{2 pi i k rates[j]/Nf} and z^16 are evaluated
// directly (k*rate/Nf reduced in FP64), and the polynomial is evaluated as
// 16-term Horner blocks combined by Horner in z^16, so no power of a rounded
// z above the 15th enters the sum.  For Nt > 64 (NT = 0) every term's phase is
// evaluated directly.
//
// COL: F and Ys in the fused output's order (bin k2 + N2 k1 at k1 + N1 k2, the
// Nyquist bins apart), else natural.  The rates are kernel arguments (no copy to
// the device to wait for), and groups of them go over blockIdx.y up to 16 wavefronts a CU.
// VALU-bound at 16 steps (about 115 operations a bin and rate): 2^18 x 16 x 64
// 29 -> 25 us.
template <int NT, bool COL>
__global__ __launch_bounds__(256) void czt_rates(CztRatesArgs a) {
  constexpr int B = NT < 16 ? (NT < 1 ? 1 : NT) : 16;
  constexpr int NB = NT / B;
  const int64_t g = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const bool in = COL || g < a.n;  // COL: whole blocks
  const int64_t o = in ? g : a.n - 1;
  const int64_t k = COL ? (g >> a.logN1) + ((g & ((int64_t(1) << a.logN1) - 1)) << a.logN2) : o;
  const double kd = static_cast<double>(k);
  const int j0 = group_first(a.Nr, blockIdx.y, gridDim.y), j1 = group_first(a.Nr, blockIdx.y + 1, gridDim.y);
  if constexpr (NT > 0) {
    c32 c[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) c[t] = (t < a.Nt) ? a.F[o + t * a.fs] : c32{0.0f, 0.0f};
#pragma unroll 2
    for (int j = j0; j < j1; ++j) {
      const c32 zf = cis_nh(kd, a.rh[j]);  // rh[j] = rates[j]/Nf
      const c32 zBf = cis_nh(kd * static_cast<double>(B), a.rh[j]);
      c32 acc = {0.0f, 0.0f};
#pragma unroll
      for (int b = NB - 1; b >= 0; --b) {
        c32 p = c[b * B + B - 1];
#pragma unroll
        for (int u = B - 2; u >= 0; --u) p = cfma(c[b * B + u], p, zf);
        acc = (b == NB - 1) ? p : cfma(p, acc, zBf);
      }
      if (in) a.Ys[o + j * a.ys] = acc;
    }
  } else {
    for (int j = j0; j < j1; ++j) {
      c32 acc = {0.0f, 0.0f};
      for (int t = 0; t < a.Nt; ++t)
        acc = cfma(acc, a.F[o + t * a.fs], cis_nh(kd * static_cast<double>(t), a.rh[j]));
      if (in) a.Ys[o + j * a.ys] = acc;
    }
  }
  if constexpr (COL) {
    // the Nyquist bin, a wavefront per rate over all blocks
    const int lane = threadIdx.x & 63, nw = 4 * gridDim.x * gridDim.y;
    for (int j = 4 * (blockIdx.y * gridDim.x + blockIdx.x) + (threadIdx.x >> 6); j < a.Nr; j += nw) {
      c32 s = {0.0f, 0.0f};
      for (int t = lane; t < a.Nt; t += 64)
        s = cfma(s, a.F[a.n * a.Nt + t], cis_nh(static_cast<double>(a.n) * static_cast<double>(t), a.rh[j]));
#pragma unroll
      for (int x = 32; x > 0; x >>= 1) {
        s.x += __shfl_xor(s.x, x, 64);
        s.y += __shfl_xor(s.y, x, 64);
      }
      if (lane == 0) a.yM[j] = s;
    }
  }
}

int launch_czt_rates(CztRatesArgs a, const double* rates_over_nf, int64_t Nr, hipStream_t st) {
  ProfScope ps(st, "czt_rates", 8.0 * static_cast<double>(a.n) * static_cast<double>(a.Nt + Nr));
  int ncu = 256, dev = 0;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  const bool col = a.yM != nullptr;
  const int nblk = static_cast<int>((a.n + 255) / 256);
  for (int64_t j0 = 0; j0 < Nr; j0 += CZT_RATES_MAX) {
    a.Nr = static_cast<int>(std::min<int64_t>(CZT_RATES_MAX, Nr - j0));
    for (int j = 0; j < a.Nr; ++j) a.rh[j] = rates_over_nf[j0 + j];
    const dim3 grid(static_cast<unsigned>(nblk), group_parts(a.Nr, nblk, 256, 16, 8, ncu));
#define ZDT_RATES(NT)                              \
  (col ? czt_rates<NT, true><<<grid, 256, 0, st>>>(a) : czt_rates<NT, false><<<grid, 256, 0, st>>>(a))
    if (a.Nt <= 4) ZDT_RATES(4);
    else if (a.Nt <= 16) ZDT_RATES(16);
    else if (a.Nt <= 32) ZDT_RATES(32);
    else if (a.Nt <= 64) ZDT_RATES(64);
    else ZDT_RATES(0);
#undef ZDT_RATES
    ZDT_CHECK_LAUNCH("czt_rates");
    a.Ys += a.Nr * a.ys;
    if (col) a.yM += a.Nr;
  }
  return ZDT_OK;
}

// fdshift (src/fftfdr.jl:104-111): Y[k,t] = F[k,t] e^{2 pi i k t rate/Nf}
__global__ __launch_bounds__(256) void shift_phase(const c32* __restrict__ F, int64_t ldF, c32* __restrict__ Y,
                                                   int64_t ldY, int64_t Nk, int Nt, double rh) {
  const int64_t total = Nk * Nt;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < total;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t k = g % Nk, t = g / Nk;
    Y[k + t * ldY] = cmul(F[k + t * ldF], cis_nh(static_cast<double>(k) * static_cast<double>(t), rh));
  }
}

int launch_shift_phase(const c32* F, int64_t ldF, c32* Y, int64_t ldY, int64_t Nk, int Nt, double rate_over_nf,
                       hipStream_t st) {
  int64_t g = (Nk * Nt + 255) / 256;
  if (g > (1 << 20)) g = 1 << 20;
  shift_phase<<<static_cast<unsigned>(g), 256, 0, st>>>(F, ldF, Y, ldY, Nk, Nt, rate_over_nf);
  ZDT_CHECK_LAUNCH("shift_phase");
  return ZDT_OK;
}

// ---------------------------------------------------------------------------
// step functions (materialized Y, src/zdtfdr.jl:221-321)
// ---------------------------------------------------------------------------

// preprocess!: Y[:, :Nt] = F .* prephase, Y[:, Nt:] = 0   (src/zdtfdr.jl:221-235)
__global__ __launch_bounds__(256) void step_prephase(const c32* __restrict__ F, int64_t ldF,
                                                     c32* __restrict__ Y, int64_t ldY, int64_t Nk,
                                                     int Nt, int Nl, double hd, double h0) {
  const int64_t total = Nk * Nl;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < total;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t k = g % Nk;
    const int t = static_cast<int>(g / Nk);
    c32 v = {0.0f, 0.0f};
    if (t < Nt) {
      const double kd = static_cast<double>(k), td = static_cast<double>(t);
      v = cmul(F[k + t * ldF], cis_sum2(kd * td * td, hd, kd * td, h0));
    }
    Y[k + t * ldY] = v;
  }
}

// chirp kernel before its FFT, in FP64 (src/zdtfdr.jl:173-185):
// V0[k,l] = chirp(k,l) for l < Nr, chirp(k, Nl-l) for l >= Nl-Nt+1, else 0
__global__ __launch_bounds__(256) void step_vgen(c64* __restrict__ V, int64_t Nk, int Nt, int Nr, int Nl,
                                                 double hd) {
  const int64_t total = Nk * Nl;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < total;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t k = g % Nk;
    const int l = static_cast<int>(g / Nk);
    c64 v = {0.0, 0.0};
    int lag = -1;
    if (l < Nr) {
      lag = l;
    } else if (l >= Nl - Nt + 1) {
      lag = Nl - l;
    }
    if (lag >= 0) {
      const double kd = static_cast<double>(k), ld = static_cast<double>(lag);
      v = cis64(-(kd * ld * ld) * hd);
    }
    V[g] = v;
  }
}

__global__ __launch_bounds__(256) void c64_to_c32(const c64* __restrict__ in, c32* __restrict__ out,
                                                  int64_t n) {
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < n;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    out[g] = {static_cast<float>(in[g].x), static_cast<float>(in[g].y)};
  }
}

// Y .*= V  (src/zdtfdr.jl:251)
__global__ __launch_bounds__(256) void step_vmul(c32* __restrict__ Y, const c32* __restrict__ V, int64_t n) {
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < n;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    Y[g] = cmul(Y[g], V[g]);
  }
}

// postprocess!: Ys .*= postphase .* w  (src/zdtfdr.jl:297-321)
__global__ __launch_bounds__(256) void step_postphase(c32* __restrict__ Y, int64_t ldY, int64_t Nk,
                                                      int64_t Nf, int Nr, double hd, int wkind,
                                                      const float* __restrict__ wcustom, float scale) {
  const int64_t total = Nk * Nr;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < total;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t k = g % Nk;
    const int j = static_cast<int>(g / Nk);
    const double kd = static_cast<double>(k), jd = static_cast<double>(j);
    double p = (kd * jd * jd) * hd;
    p -= __builtin_rint(p);
    const c32 post = cis_rev(static_cast<float>(p));
    const float w = window_value(wkind, wcustom, k, Nf) * scale;
    c32 v = cmul(Y[k + j * ldY], post);
    Y[k + j * ldY] = {v.x * w, v.y * w};
  }
}

static unsigned grid_for(int64_t total) {
  int64_t g = (total + 255) / 256;
  if (g > (1 << 20)) g = 1 << 20;
  if (g < 1) g = 1;
  return static_cast<unsigned>(g);
}

int launch_step_prephase(const c32* F, int64_t ldF, c32* Y, int64_t ldY, int64_t Nk, int Nt, int Nl,
                         double hd, double h0, hipStream_t st) {
  ProfScope ps(st, "step_prephase", 8.0 * static_cast<double>(Nk) * (Nt + Nl));
  step_prephase<<<grid_for(Nk * Nl), 256, 0, st>>>(F, ldF, Y, ldY, Nk, Nt, Nl, hd, h0);
  ZDT_CHECK_LAUNCH("step_prephase");
  return ZDT_OK;
}

int launch_step_vgen(c64* V, int64_t Nk, int Nt, int Nr, int Nl, double hd, hipStream_t st) {
  step_vgen<<<grid_for(Nk * Nl), 256, 0, st>>>(V, Nk, Nt, Nr, Nl, hd);
  ZDT_CHECK_LAUNCH("step_vgen");
  return ZDT_OK;
}

int launch_c64_to_c32(const c64* in, c32* out, int64_t n, hipStream_t st) {
  c64_to_c32<<<grid_for(n), 256, 0, st>>>(in, out, n);
  ZDT_CHECK_LAUNCH("c64_to_c32");
  return ZDT_OK;
}

int launch_step_vmul(c32* Y, const c32* V, int64_t n, hipStream_t st) {
  ProfScope ps(st, "step_vmul", 24.0 * static_cast<double>(n));
  step_vmul<<<grid_for(n), 256, 0, st>>>(Y, V, n);
  ZDT_CHECK_LAUNCH("step_vmul");
  return ZDT_OK;
}

int launch_step_postphase(c32* Y, int64_t ldY, int64_t Nk, int64_t Nf, int Nr, double hd, int wkind,
                          const float* wcustom, float scale, hipStream_t st) {
  ProfScope ps(st, "step_postphase", 16.0 * static_cast<double>(Nk * Nr));
  step_postphase<<<grid_for(Nk * Nr), 256, 0, st>>>(Y, ldY, Nk, Nf, Nr, hd, wkind, wcustom, scale);
  ZDT_CHECK_LAUNCH("step_postphase");
  return ZDT_OK;
}

}  // namespace zdt
