// The chirp-Z sum of a bin for a mirrored pair of rates, folded about the
// middle of 16-step blocks of time:
//   Y(z) = sum_t c_t z^t and Y(conj z), z = e^{i theta},
// with the block's middle factored out,
//   sum_{t=16q}^{16q+15} c_t z^t = z^{16q} z^{7.5} (A_q + i B_q),
//   A_q = sum_s (c_{m+s} + c_{m-s}) cos(s theta),  B_q = sum_s (c_{m+s} - c_{m-s}) sin(s theta),
// m = 16q + 7.5, s = 1/2, 3/2, .., 15/2; conj(z) changes the sign of B_q and
// conjugates the powers.  The sums and differences are made once per bin, so
// a pair of rates costs 32 real FMAs per block (two per time step, against
// six operations for the Reinsch recurrence and eight for two complex Horner
// sums), 12 operations to combine a block (Horner in z^16), and once per pair
// the eight powers z^s: z^{1/2} and z from FP64, z^{3/2} .. z^{7/2} by complex
// multiplies, the upper four by cos((4+x)a) = 2 cos 4a cos xa - cos((4-x)a)
// and the like for sin.  No recurrence runs over the time steps, so the error
// does not grow with them: FP32 emulation over random angles (down to 1e-6
// from 0 and pi) gives 6.6e-8 rms of sum|c_t| for coherent coefficients at
// 16, 32 and 64 steps, where Reinsch gives 8e-8, 1.5e-7 and 2.7e-7.  Sums of 6 to
// 15 steps are centred in their block, so that s stays small, and up to 5 are
// Horner sums in z: against uniform angles and independent coefficients, rms of the
// result, 4 steps 6.2e-8 (Reinsch 6.7e-8), 6 7.7e-8 (8.2e-8), 10 9.4e-8 (1.1e-7), where
// a block that starts at step 0 gives 1.2e-7 for all of them.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "rate_groups.h"
#include "zdt_internal.h"

namespace zdt {

constexpr int FOLD = 16;  // time steps per block

// z^2 for |z| = 1
__device__ __forceinline__ c64 unit_sq(c64 z) {
  const double y2 = z.y + z.y;
  return {__builtin_fma(-y2, z.y, 1.0), z.x * y2};
}

// exp(2 pi i rev) in FP64
__device__ __forceinline__ c64 cis64f(double rev) {
  const double f = rev - __builtin_rint(rev);
  double s, c;
  sincospi(2.0 * f, &s, &c);
  return {c, s};
}

// cis_nh without branches, for the many phases of a bin's pre-rotation: odd
// quarter turns swap the parts, turns 1 and 2 negate the real one, 2 and 3 the
// imaginary one
__device__ __forceinline__ c32 cis_nh_flat(double n, double h) {
  const double p = n * h;
  const float f = static_cast<float>(p - __builtin_rint(p));
  const float q = __builtin_rintf(4.0f * f);
  float s, c;
  sincos_2pi_small(__builtin_fmaf(q, -0.25f, f), &s, &c);
  const unsigned iq = static_cast<unsigned>(static_cast<int>(q));
  const float a = (iq & 1u) ? s : c, b = (iq & 1u) ? c : s;
  return {__uint_as_float(__float_as_uint(a) ^ (((iq + 1u) & 2u) << 30)),
          __uint_as_float(__float_as_uint(b) ^ ((iq & 2u) << 30))};
}

__device__ __forceinline__ c32 to_c32(c64 z) { return {static_cast<float>(z.x), static_cast<float>(z.y)}; }

// Sums and differences of the coefficients about the block middles:
// p[q][i] = c_{16q+8+i} + c_{16q+7-i}, m[q][i] = c_{16q+8+i} - c_{16q+7-i}
template <int NB>
struct FoldCoef {
  c32 p[NB][FOLD / 2], m[NB][FOLD / 2];

  // raw(t): the input of time step t, called for all steps in order
  // before coef(t, input) turns the first of them into its coefficient, so
  // that the loads are in flight together
  template <typename Raw, typename Coef>
  __device__ __forceinline__ void load(Raw&& raw, Coef&& coef) {
#pragma unroll
    for (int t = 0; t < FOLD * NB; ++t) {
      const c32 v = raw(t);
      if (t % FOLD >= FOLD / 2)
        p[t / FOLD][t % FOLD - FOLD / 2] = v;
      else
        m[t / FOLD][FOLD / 2 - 1 - t % FOLD] = v;
    }
#pragma unroll
    for (int q = 0; q < NB; ++q)
#pragma unroll
      for (int i = 0; i < FOLD / 2; ++i) {
        const c32 hi = coef(FOLD * q + FOLD / 2 + i, p[q][i]), lo = coef(FOLD * q + FOLD / 2 - 1 - i, m[q][i]);
        p[q][i] = cadd(hi, lo);
        m[q][i] = csub(hi, lo);
      }
  }
};

// The powers of z = e^{i theta} a pair of rates needs, rounded from FP64:
// h = z^{1/2}, z, 2 cos 4 theta, z^{7.5} and (for more than one block) z^16.
struct FoldPow {
  c32 h, z, z75, z16;
  float c4;
};

template <int NB>
__device__ __forceinline__ FoldPow fold_powers(c64 h) {
  FoldPow w;
  const c64 z1 = unit_sq(h), z4 = unit_sq(unit_sq(z1)), z8 = unit_sq(z4);
  w.h = to_c32(h);
  w.z = to_c32(z1);
  w.c4 = 2.0f * static_cast<float>(z4.x);
  w.z75 = cmulc(to_c32(z8), w.h);
  w.z16 = NB > 1 ? to_c32(unit_sq(z8)) : c32{1.0f, 0.0f};
  return w;
}

// U = sum_q z^{16q} (A_q + i B_q) and V the same at conj z: Y(z) = z^{7.5} U,
// Y(conj z) = conj(z^{7.5}) V.
template <int NB>
__device__ __forceinline__ void fold_sums(const FoldCoef<NB>& c, const FoldPow& w, c32& U, c32& V) {
  c32 P[FOLD / 2];
  P[0] = w.h;
#pragma unroll
  for (int i = 1; i < 4; ++i) P[i] = cmul(P[i - 1], w.z);
#pragma unroll
  for (int i = 0; i < 4; ++i) P[4 + i] = {fmaf(w.c4, P[i].x, -P[3 - i].x), fmaf(w.c4, P[i].y, P[3 - i].y)};
#pragma unroll
  for (int q = NB - 1; q >= 0; --q) {
    float Ar = c.p[q][0].x * P[0].x, Ai = c.p[q][0].y * P[0].x;
    float Br = c.m[q][0].x * P[0].y, Bi = c.m[q][0].y * P[0].y;
#pragma unroll
    for (int i = 1; i < FOLD / 2; ++i) {
      Ar = fmaf(c.p[q][i].x, P[i].x, Ar);
      Ai = fmaf(c.p[q][i].y, P[i].x, Ai);
      Br = fmaf(c.m[q][i].x, P[i].y, Br);
      Bi = fmaf(c.m[q][i].y, P[i].y, Bi);
    }
    const c32 u = {Ar - Bi, Ai + Br}, v = {Ar + Bi, Ai - Br};
    U = q == NB - 1 ? u : cfma(u, U, w.z16);
    V = q == NB - 1 ? v : cfma(v, V, cconj(w.z16));
  }
}

__device__ __forceinline__ void store_past(c32* p, c32 v) {
  typedef float f2v __attribute__((ext_vector_type(2)));
  __builtin_nontemporal_store(f2v{v.x, v.y}, reinterpret_cast<f2v*>(p));
}

// A bin's chirp-Z over a range of rate pairs.  F, dst and their steps are
// uniform over the block, so that only the bin's offset takes a vector register.
struct FoldBin {
  const c32* F;    // input spectrum, time step 0
  int64_t fs;      // its step in t
  c32* dst;        // Ys, rate 0
  int64_t stride;  // its step in rate
  unsigned o;      // the bin's offset in both
  double kd;       // the bin k
  float w;         // window weight and scale
  int* wide;       // fold_rates<NB, NC, true>: NULL, or set where the coefficients pass FOLD_WIDE
};

// Bound on the sum of a lane's coefficients |Re| + |Im| under which spectra of up
// to 2^20 time steps stay below 2^96, and sums over 2^20 of them far from overflow.
constexpr float FOLD_WIDE = 1.2e24f;  // 2^80

struct FoldRates {
  int Nt, Nr;
  double hd2;  // dr/Nf
  double hc;   // rc/Nf, rc = r0 + (Nr-1) dr/2: the pre-rotation by the centre rate
  double hz;   // (r0 - rc)/Nf
};

// v of the lane whose index differs in bit 0 (X = 1) or bit 1 (X = 2)
template <int X>
__device__ __forceinline__ float quad_xor(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), X == 1 ? 0xb1 : 0x4e, 0xf, 0xf, false));
}

// y into rate j and yc into rate jp, unless they are one (see fold_rates)
__device__ __forceinline__ void fold_store(const FoldBin& b, int j, int jp, c32 y, c32 yc, bool acc, bool past) {
  c32* dj = b.dst + static_cast<int64_t>(j) * b.stride;   // uniform
  c32* dp = b.dst + static_cast<int64_t>(jp) * b.stride;  // uniform
  if (acc) {
    y = cadd(y, dj[b.o]);
    if (jp != j) yc = cadd(yc, dp[b.o]);
  }
  if (past) {  // uniform
    store_past(dj + b.o, y);
    if (jp != j) store_past(dp + b.o, yc);
  } else {
    dj[b.o] = y;
    if (jp != j) dp[b.o] = yc;
  }
}

// fold_rates for up to FOLD_SHORT time steps: Horner in z and conj z
constexpr int FOLD_SHORT = 5;
template <bool GUARD>
__device__ __forceinline__ void short_rates(const FoldBin& b, const FoldRates& r, int jlo, int jhi, bool past) {
  c32 c[FOLD_SHORT];
#pragma unroll
  for (int t = 0; t < FOLD_SHORT; ++t) c[t] = (b.F + static_cast<int64_t>(min(t, r.Nt - 1)) * b.fs)[b.o];
#pragma unroll
  for (int t = 0; t < FOLD_SHORT; ++t) {
    c32 v = c[t];
    if (r.hc != 0.0) v = cmul(v, cis_nh_flat(b.kd * static_cast<double>(t), r.hc));  // uniform
    c[t] = t < r.Nt ? c32{v.x * b.w, v.y * b.w} : c32{0.0f, 0.0f};
  }
  const double hs = r.hz + static_cast<double>(jlo) * r.hd2;
  c64 z = cis64f(b.kd * hs);
  const c64 g = cis64f(b.kd * r.hd2);
  for (int j = jlo; j < jhi; ++j) {
    const c32 w = to_c32(z), wc = cconj(w);
    z = cmul(z, g);
    c32 y = c[FOLD_SHORT - 1], yc = y;
#pragma unroll
    for (int t = FOLD_SHORT - 2; t >= 0; --t) {
      y = cfma(c[t], y, w);
      yc = cfma(c[t], yc, wc);
    }
    fold_store(b, j, r.Nr - 1 - j, y, yc, false, past);
  }
  if (GUARD && b.wide != nullptr) {  // uniform
    float mag = 0.0f;
#pragma unroll
    for (int t = 0; t < FOLD_SHORT; ++t) mag += fabsf(c[t].x) + fabsf(c[t].y);
    if (!(mag < FOLD_WIDE)) *b.wide = 1;
  }
}

// Rates j in [jlo, jhi) and their mirrors Nr-1-j (the middle rate of an odd Nr
// is its own), j < (Nr+1)/2.  NC adjacent lanes share a bin: lane q sums the
// time steps t0 .. t0 + 16 NB - 1, t0 = tbase + 16 NB q, and the NC partial
// sums are added with each lane keeping a share (with four lanes and more: one
// of the two rates by its bit 0, the real or imaginary part by its bit 1), so
// a pair takes log2(NC) + 1 exchanges.  acc: add to what dst holds.  past
// (one lane per bin): store past the last-level cache (nontemporal), for
// destinations larger than it whose rows are whole cache lines; on rows that are
// not, such stores cost half as much again (10^6 channels x 129: 136 -> 192 us).
// GUARD: set *b.wide, if there is one, where the coefficients reach FOLD_WIDE or
// are not finite.
template <int NB, int NC, bool GUARD = false>
__device__ __forceinline__ void fold_rates(const FoldBin& b, const FoldRates& r, int q, int tbase, int jlo, int jhi,
                                           bool acc, bool past) {
  // the first time step; a sum that fits one block is centred in it
  const int t0 = tbase + FOLD * NB * q - (NB == 1 ? max(0, (FOLD - (r.Nt - tbase)) / 2) : 0);
  FoldCoef<NB> c;
  // the time step's input; outside the steps the nearest one again, dropped below
  const c32* f = b.F + static_cast<int64_t>(min(t0, r.Nt - 1)) * b.fs;
  c.load(
      [&](int i) {
        if constexpr (NC == 1) {
          return (b.F + static_cast<int64_t>(max(min(t0 + i, r.Nt - 1), 0)) * b.fs)[b.o];  // uniform base
        } else {
          const c32 v = f[b.o];
          f += t0 + i + 1 < r.Nt ? b.fs : 0;
          return v;
        }
      },
      [&](int i, c32 v) {
        const int t = t0 + i;
        if (r.hc != 0.0) v = cmul(v, cis_nh_flat(b.kd * static_cast<double>(t), r.hc));  // uniform
        return (NB > 1 || t >= tbase) && t < r.Nt ? c32{v.x * b.w, v.y * b.w} : c32{0.0f, 0.0f};
      });
  const double hs = r.hz + static_cast<double>(jlo) * r.hd2;  // (r_jlo - rc)/Nf
  // h = z^{1/2} and its step between rates.  With four and five blocks they wait
  // in LDS: their eight registers would spill beside 128 of coefficients at
  // three wavefronts per SIMD
  constexpr bool PARK = NB >= 4;
  __shared__ c64 state[2][PARK ? 256 : 1];
  c64 h = cis64f(0.5 * b.kd * hs), g = cis64f(0.5 * b.kd * r.hd2);
  if constexpr (PARK) {
    state[0][threadIdx.x] = h;
    state[1][threadIdx.x] = g;
  }
  // the lane's place in the sum: z^{t0}, by a recurrence of its own (one block: z^{t0 + 7.5})
  constexpr bool ONE = NB == 1 && NC == 1;
  const bool placed = ONE || NC > 1 || tbase > 0;
  const double td = static_cast<double>(t0) + (ONE ? 7.5 : 0.0);
  c64 gq = {1.0, 0.0}, zq = {1.0, 0.0};
  if (placed) {
    gq = cis64f(b.kd * r.hd2 * td);
    zq = cis64f(b.kd * hs * td);
  }
  for (int j = jlo; j < jhi; ++j) {
    const int jp = r.Nr - 1 - j;
    int me = static_cast<int>(threadIdx.x);
    if constexpr (PARK) {
      asm volatile("" : "+v"(me));  // read and written here, not carried in registers
      h = state[0][me];
    }
    const FoldPow w = fold_powers<NB>(h);
    if constexpr (PARK)
      state[0][me] = cmul(h, state[1][me]);
    else
      h = cmul(h, g);
    c32 U, V, z75 = w.z75;
    if (placed) {
      z75 = ONE ? to_c32(zq) : cmul(z75, to_c32(zq));
      zq = cmul(zq, gq);
    }
    fold_sums<NB>(c, w, U, V);
    const c32 y = cmul(U, z75), yc = cmulc(V, z75);
    if constexpr (NC == 1) {
      fold_store(b, j, jp, y, yc, acc, past);
    } else {
      c32* dj = b.dst + static_cast<int64_t>(j) * b.stride;   // uniform
      c32* dp = b.dst + static_cast<int64_t>(jp) * b.stride;  // uniform
      // bit 0 keeps y (0) or yc (1)
      const bool b0 = q & 1;
      const float kx = b0 ? yc.x : y.x, ky = b0 ? yc.y : y.y;
      const float gx = b0 ? y.x : yc.x, gy = b0 ? y.y : yc.y;
      c32 k = {kx + quad_xor<1>(gx), ky + quad_xor<1>(gy)};
      c32* d = (b0 ? dp : dj) + b.o;
      const bool mine = !b0 || jp != j;
      if constexpr (NC == 2) {
        if (mine) *d = acc ? cadd(k, *d) : k;
      } else {
        // bit 1 keeps the real (0) or imaginary (1) part
        const bool b1 = q & 2;
        const float keep = b1 ? k.y : k.x, give = b1 ? k.x : k.y;
        float v = keep + quad_xor<2>(give);
#pragma unroll
        for (int x = 4; x < NC; x <<= 1) v += __shfl_xor(v, x, 64);
        float* df = reinterpret_cast<float*>(d) + (b1 ? 1 : 0);
        if (mine && q < 4) *df = acc ? v + *df : v;
      }
    }
  }
  // last, so that nothing above waits for the coefficients any sooner
  if (GUARD && b.wide != nullptr) {  // uniform
    float mag = 0.0f;  // at least the sum over the coefficients
#pragma unroll
    for (int u = 0; u < NB; ++u)
#pragma unroll
      for (int i = 0; i < FOLD / 2; ++i) {
        mag += fabsf(c.p[u][i].x) + fabsf(c.p[u][i].y);
        mag += fabsf(c.m[u][i].x) + fabsf(c.m[u][i].y);
      }
    if (!(mag < FOLD_WIDE)) *b.wide = 1;
  }
}

// Lanes per bin and blocks per lane for Nt time steps: up to five blocks (160
// coefficient registers, two wavefronts per SIMD) stay in one lane, because
// the powers (about 70 operations a pair) are made by every lane of a bin.
// At most FOLD_MAX_NC lanes: FOLD_MAX_NT steps in one go.
constexpr int FOLD_MAX_NB = 5, FOLD_MAX_NC = 16;
constexpr int FOLD_MAX_NT = FOLD * FOLD_MAX_NB * FOLD_MAX_NC;

// Whether the chirp-Z of `bytes` of spectra with nb blocks per bin stores past
// the last-level cache: spectra that fit half of it are read from it next, and
// from four blocks on the VALU sets the pace (2^22 x 64 x 257: 1556 us through
// the cache, 1610 past it; 2^22 x 16 x 65 270 and 229).
inline bool fold_past(int64_t bytes, int nb) { return bytes > (int64_t(128) << 20) && nb < 4; }

// No block (short_rates) for a whole sum of up to FOLD_SHORT steps.
inline void fold_split(int64_t Nt, int64_t tbase, int* nb, int* nc) {
  const int n = Nt <= FOLD_SHORT ? 0 : static_cast<int>((Nt - tbase + FOLD - 1) / FOLD);
  *nc = 1;
  while (*nc < FOLD_MAX_NC && n > FOLD_MAX_NB * *nc) *nc *= 2;
  *nb = n >= FOLD_MAX_NB * FOLD_MAX_NC ? FOLD_MAX_NB : (n + *nc - 1) / *nc;
}

// f.template operator()<NB, NC>() for the (nb, nc) of fold_split
template <typename Fn>
bool fold_dispatch(int nb, int nc, Fn&& f) {
#define ZDT_FOLD_CASE(B, C)      \
  case B * 32 + C:               \
    f(std::integral_constant<int, B>(), std::integral_constant<int, C>()); \
    return true;
  switch (nb * 32 + nc) {
    ZDT_FOLD_CASE(0, 1)
    ZDT_FOLD_CASE(1, 1)
    ZDT_FOLD_CASE(2, 1)
    ZDT_FOLD_CASE(3, 1)
    ZDT_FOLD_CASE(4, 1)
    ZDT_FOLD_CASE(5, 1)
    ZDT_FOLD_CASE(3, 2)
    ZDT_FOLD_CASE(4, 2)
    ZDT_FOLD_CASE(5, 2)
    ZDT_FOLD_CASE(3, 4)
    ZDT_FOLD_CASE(4, 4)
    ZDT_FOLD_CASE(5, 4)
    ZDT_FOLD_CASE(3, 8)
    ZDT_FOLD_CASE(4, 8)
    ZDT_FOLD_CASE(5, 8)
    ZDT_FOLD_CASE(3, 16)
    ZDT_FOLD_CASE(4, 16)
    ZDT_FOLD_CASE(5, 16)
    default:
      return false;
  }
#undef ZDT_FOLD_CASE
}

}  // namespace zdt
