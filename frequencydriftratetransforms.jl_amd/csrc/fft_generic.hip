// Generic batched mixed-radix FFT for gfx950 (FP32 and FP64).
//
// This engine serves every transform whose size or layout the fused ZDT path
// does not cover: the step functions' length-Nl FFT along dim 2 of the Nk x Nl
// work matrix (src/zdtfdr.jl:122-123,186,250-252), the chirp-kernel spectrum V
// (computed in FP64, src/zdtfdr.jl:173-187), and the frequency-axis r2c/c2r of
// the generic path (src/zdtfdr.jl:119-120,211,330) for any Nf whose prime
// factors are in {2,3,5,7,11,13}.
//
// Algorithm: Stockham auto-sort, one kernel per radix pass, in the
// formulation of Govindaraju et al., "High performance discrete Fourier
// transforms on graphics processors" (SC'08): pass with radix R over the
// current sub-transform length Ns reads x[j + r*N/R], applies the twiddles
// W_{Ns*R}^{r*(j mod Ns)}, does a length-R DFT and writes
// y[(j/Ns)*Ns*R + (j mod Ns) + r*Ns].  Twiddles come from a per-N FP64-derived
// table W_N^m.  The inverse is conj(forward(conj(x))).  The thread order is
// chosen so that consecutive lanes touch consecutive addresses: along j when
// the transform axis is contiguous, along the batch otherwise.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <vector>

#include "fft_butterflies.h"
#include "fft_generic.h"

namespace zdt {

// ---------------------------------------------------------------- pass kernel

struct PassArgs {
  int64_t N, NR, Ns, twstep;  // twstep = N/(Ns*R)
  int64_t ies, ibs, oes, obs, batch;
  double scale;
  int inverse, jmajor;
};

template <typename T, int R>
__global__ __launch_bounds__(256) void stockham_pass(const cplx<T>* __restrict__ in,
                                                     cplx<T>* __restrict__ out,
                                                     const cplx<T>* __restrict__ tw, PassArgs a) {
  const int64_t total = a.NR * a.batch;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < total;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    int64_t j, b;
    if (a.jmajor) {
      j = g % a.NR;
      b = g / a.NR;
    } else {
      b = g % a.batch;
      j = g / a.batch;
    }
    const int64_t k = j % a.Ns;
    cplx<T> v[R];
    const cplx<T>* src = in + b * a.ibs;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      v[r] = src[(j + r * a.NR) * a.ies];
      if (a.inverse) v[r].y = -v[r].y;
    }
    if (a.Ns > 1) {
#pragma unroll
      for (int r = 1; r < R; ++r) v[r] = cmul(v[r], tw[r * k * a.twstep]);
    }
    dft<T, R>(v);
    const T sc = static_cast<T>(a.scale);
    const int64_t idxD = (j / a.Ns) * a.Ns * R + k;
    cplx<T>* dst = out + b * a.obs;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      cplx<T> y = v[r];
      if (a.inverse) y.y = -y.y;
      if (a.scale != 1.0) y = {y.x * sc, y.y * sc};
      dst[(idxD + r * a.Ns) * a.oes] = y;
    }
  }
}

static unsigned grid_for(int64_t total, int threads) {
  int64_t g = (total + threads - 1) / threads;
  if (g > (1 << 20)) g = 1 << 20;
  if (g < 1) g = 1;
  return static_cast<unsigned>(g);
}

template <typename T>
static int launch_pass(int R, const cplx<T>* in, cplx<T>* out, const cplx<T>* tw, const PassArgs& a,
                       hipStream_t st) {
  const unsigned grid = grid_for(a.NR * a.batch, 256);
  static const char* names[17] = {nullptr, nullptr, "fft_pass_r2", "fft_pass_r3", "fft_pass_r4", "fft_pass_r5",
                                  nullptr, "fft_pass_r7", "fft_pass_r8", nullptr, nullptr, "fft_pass_r11",
                                  nullptr, "fft_pass_r13", nullptr, nullptr, "fft_pass_r16"};
  ProfScope ps(st, (R >= 2 && R <= 16 && names[R]) ? names[R] : "fft_pass",
               2.0 * static_cast<double>(a.N * a.batch) * sizeof(cplx<T>));
#define ZDT_PASS_CASE(RR)                                                  \
  case RR:                                                                 \
    stockham_pass<T, RR><<<grid, 256, 0, st>>>(in, out, tw, a);            \
    break;
  switch (R) {
    ZDT_PASS_CASE(2)
    ZDT_PASS_CASE(3)
    ZDT_PASS_CASE(4)
    ZDT_PASS_CASE(5)
    ZDT_PASS_CASE(7)
    ZDT_PASS_CASE(8)
    ZDT_PASS_CASE(11)
    ZDT_PASS_CASE(13)
    ZDT_PASS_CASE(16)
    default:
      return fail(ZDT_ENOTSUP, "internal: radix %d not implemented", R);
  }
#undef ZDT_PASS_CASE
  ZDT_CHECK_LAUNCH("stockham_pass");
  return ZDT_OK;
}

template <typename T>
__global__ __launch_bounds__(256) void scale_copy(const cplx<T>* __restrict__ in, int64_t ibs,
                                                  cplx<T>* __restrict__ out, int64_t obs, int64_t batch,
                                                  T scale) {
  for (int64_t b = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; b < batch;
       b += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const cplx<T> v = in[b * ibs];
    out[b * obs] = {v.x * scale, v.y * scale};
  }
}

static int pow2_floor(int64_t x) {
  int r = 1;
  while (static_cast<int64_t>(r) * 2 <= x) r *= 2;
  return r;
}

// ---------------------------------------------------------------- transforms in LDS
//
// FP32 transforms along a contiguous axis run as Stockham passes on one LDS
// buffer: each pass reads its butterflies' inputs into registers, synchronizes,
// and writes the outputs in place.  N <= FS_ONE takes one kernel (fs_one, T
// transforms a block).  Longer ones with N = N1 * N2 (N1 <= 1024, N2 <= 2048, N <=
// 2^20) take two kernels that each move the data through HBM once (the
// "four-step" FFT, D. H. Bailey, "FFTs in external or hierarchical memory", 1990):
//   fs_cols  X1[n2 + N2 k1] = W_N^{n2 k1} sum_{n1} x[n2 + N2 n1] W_N1^{n1 k1}
//            (TC adjacent columns n2 per block, so loads and stores are
//            TC-element runs)
//   fs_rows  X[k1 + N1 k2] = sum_{n2} X1[n2 + N2 k1] W_N2^{n2 k2}
//            (TR adjacent rows k1 per block; the stores are TR-element runs)
// A pass reads its twiddles W_{Ns R}^{r k} from a table of its own in LDS
// (contiguous or broadcast reads, no products); the radices (up to 16, the
// composite ones 6, 9, 10, 12, 14, 15 among them) are chosen for the fewest
// passes.  The four-step and c2r twiddles are products of two factors evaluated
// from exact phases, the start of a thread and the step to its i-th element.  The
// inverse is conj(forward(conj(x))), conjugated on the first load and the last
// store, where the real transforms' packing happens too (fs_mode).
//
// Bound: loads, passes and stores of a block follow one another, and two blocks a
// CU (LDS) overlap them only partly; fs_rows runs its vector units 50% of the time,
// the c2r columns 65%.  Against prime radices up to 13 and 16, one twiddle table of
// the whole length in global memory and 512 threads a block with 16 elements each
// (us): Nf = 10^6, 129 rates (1.03 GB through fs_cols, as much through fs_rows)
// c2r columns 403 -> 305, rows 374 -> 278; r2c columns 59 -> 40.  Odd Nf = 99225, 77
// rates, two columns a transform instead of a zero imaginary part: 86 + 70 + 40
// for filling in the Hermitian half and taking the real part -> 39 + 42.  Nf =
// 4096, 33 rates: six launches of 5 to 6 -> two, 17 together (fs_one).  Of that, 8
// elements a thread and 1024 threads: c2r columns 318 -> 305; 32-bit offsets and
// wave-uniform strides in place of an index per access (112 -> 76 vector
// instructions an element in fs_rows): rows 295 -> 278.  Persistent blocks that load the
// next rows before the passes spill (128 VGPRs, 16 elements): 295 -> 569.  Chunks
// whose intermediate stays in the last-level cache: 0.93 to 1.0 of the speed.

constexpr int FS_PER = 8;    // elements a thread
constexpr int FS_E = 8192;   // most elements per block of fs_cols / fs_rows (TC * N1 or TR * N2)
constexpr int FS_ONE = 4096; // most elements per block of fs_one
constexpr int FS_ONE_TH = FS_ONE / FS_PER;
constexpr int FS_MAXP = 12;  // passes per sub-transform

enum fs_mode {
  FS_C2C,
  FS_C2R,      // in: half spectra X[0..N] of real sequences of length 2N; out: their N packed pairs
  FS_R2C,      // fs_one: the reverse
  FS_ODD_R2C,  // in: real sequences of odd length N; out: X[0 .. N/2]
  FS_ODD_C2R,  // in: half spectra X[0 .. N/2]; out: the real columns
};

struct FsArgs {
  const c32* in;
  int64_t ibs;  // between transforms (complex elements; floats for FS_ODD_R2C)
  c32* out;
  int64_t obs;  // (floats for FS_ODD_C2R)
  const c32* tw;
  int ntw;
  c32 half[FS_PER];  // FS_C2R of fs_cols: W_{2 N1}^{i TH / TC}
  int N, N1, N2, T;  // T = TC (fs_cols), TR (fs_rows) or transforms per block (fs_one)
  int np;            // passes of the sub-transform
  int rad[FS_MAXP];
  int inverse, mode;
  int64_t batch;     // transforms
  float scale;
  double h;          // 1/N
};

// and of the kernels with two real columns a transform (FS_ODD_C2R); apart, because
// 16 bytes more of arguments cost a 6 to 9 us kernel 0.2 us
struct FsPair {
  int64_t ncol;
  const int64_t* wide;  // not 0: one column a transform after all
};
struct FsNoPair {};
template <bool PAIR>
using FsPairOf = std::conditional_t<PAIR, FsPair, FsNoPair>;

// u / d for u * d < 2^32 by one high multiply with m = ceil(2^32 / d)
// (m = 0 marks d = 1)
struct FsDiv {
  uint32_t d, m;
};
__device__ __forceinline__ FsDiv fs_div(int d) {
  const uint32_t ud = static_cast<uint32_t>(d);
  return {ud, ud == 1 ? 0u : static_cast<uint32_t>(0xFFFFFFFFull / ud + 1)};
}
__device__ __forceinline__ int fs_quo(int u, FsDiv q) {
  return q.m == 0 ? u : static_cast<int>(__umulhi(static_cast<uint32_t>(u), q.m));
}

// element at a 32-bit byte offset: with a wave-uniform base the offset goes into
// the instruction as it is
template <typename T>
__device__ __forceinline__ T& at_byte(T* base, uint32_t off) {
  return *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + off);
}
template <typename T>
__device__ __forceinline__ const T& at_byte(const T* base, uint32_t off) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
}

// One Stockham pass of radix R over T interleaved transforms of length L
// held in buf (element n of transform c at n * T + c, T a power of two, L * T <=
// FS_PER TH).  Butterfly u covers transform c = u mod T and index j = u / T < L/R.  Every
// index is below 2^13, so j mod Ns is an exact high multiply.  tw: the pass's
// twiddles W_{Ns R}^{r k} at (r - 1) Ns + k (none in the FIRST pass, Ns = 1).
// Addresses are one start a butterfly plus wave-uniform multiples.
template <int R, int TH, bool FIRST>
__device__ __forceinline__ void fs_pass(c32* buf, const c32* tw, int L, int T, int Ns) {
  constexpr int NB = (FS_PER + R - 1) / R;
  const int Lr = L / R;
  const int nbf = Lr * T;
  const int lgT = __ffs(T) - 1;
  const FsDiv dNs = fs_div(Ns);
  const uint32_t is = 8u * static_cast<uint32_t>(nbf), os = 8u * static_cast<uint32_t>(Ns * T),
                 ws = 8u * static_cast<uint32_t>(Ns);
  // opaque to the optimizer, so that no index below is hoisted out of the
  // pass loop (which would keep every pass's indices live and spill)
  int tid = static_cast<int>(threadIdx.x);
  asm volatile("" : "+v"(tid));
  c32 v[NB][R];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int u = tid + i * TH;
    if (u < nbf) {
      const uint32_t ib = 8u * static_cast<uint32_t>(u);
#pragma unroll
      for (int r = 0; r < R; ++r) v[i][r] = at_byte(buf, ib + static_cast<uint32_t>(r) * is);
      if (!FIRST) {
        const int j = u >> lgT;
        const uint32_t kb = 8u * static_cast<uint32_t>(j - fs_quo(j, dNs) * Ns);
#pragma unroll
        for (int r = 1; r < R; ++r)
          v[i][r] = cmul(v[i][r], at_byte(tw, kb + static_cast<uint32_t>(r - 1) * ws));
      }
      dft<float, R>(v[i]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int u = tid + i * TH;
    if (u < nbf) {
      const int j = u >> lgT;
      const int q = FIRST ? j : fs_quo(j, dNs) * Ns;
      const uint32_t ob = 8u * static_cast<uint32_t>(u + ((q * (R - 1)) << lgT));
#pragma unroll
      for (int r = 0; r < R; ++r) at_byte(buf, ob + static_cast<uint32_t>(r) * os) = v[i][r];
    }
  }
  __syncthreads();
}

template <int TH, bool FIRST>
__device__ __forceinline__ void fs_pass_any(c32* buf, const c32* tw, int L, int T, int Ns, int R) {
  switch (R) {
#define ZDT_FS_CASE(RR)                        \
  case RR:                                     \
    fs_pass<RR, TH, FIRST>(buf, tw, L, T, Ns);     \
    break;
    ZDT_FS_CASE(2)
    ZDT_FS_CASE(3)
    ZDT_FS_CASE(4)
    ZDT_FS_CASE(5)
    ZDT_FS_CASE(6)
    ZDT_FS_CASE(7)
    ZDT_FS_CASE(8)
    ZDT_FS_CASE(9)
    ZDT_FS_CASE(10)
    ZDT_FS_CASE(11)
    ZDT_FS_CASE(12)
    ZDT_FS_CASE(13)
    ZDT_FS_CASE(14)
    ZDT_FS_CASE(15)
    ZDT_FS_CASE(16)
#undef ZDT_FS_CASE
  }
}

// all passes of the T interleaved sub-transforms of length L (natural order in
// and out)
template <int TH>
__device__ __forceinline__ void fs_dft(c32* buf, const c32* tw, const FsArgs& a, int L) {
  int Ns = a.rad[0];
  fs_pass_any<TH, true>(buf, tw, L, a.T, 1, Ns);
  for (int p = 1; p < a.np; ++p) {
    const int R = a.rad[p];
    fs_pass_any<TH, false>(buf, tw, L, a.T, Ns, R);
    tw += (R - 1) * Ns;
    Ns *= R;
  }
}

// the packed sequence of the c2r transform: Z[k] = E + i O with
// E = (p + conj q)/2, O = W_{2N}^{-k} (p - conj q)/2, p = X[k], q = X[N-k], w = W_{2N}^k;
// Im X[0] and Im X[N] are ignored
__device__ __forceinline__ c32 c2r_pack(int k, c32 p, c32 q, c32 w) {
  if (k == 0) return {0.5f * (p.x + q.x), 0.5f * (p.x - q.x)};
  const c32 Ev = {0.5f * (p.x + q.x), 0.5f * (p.y - q.y)};
  const c32 D = {0.5f * (p.x - q.x), 0.5f * (p.y + q.y)};
  const c32 O = cmulc(D, w);
  return {Ev.x - O.y, Ev.y + O.x};
}

// bin of the half spectrum X[0 .. N/2] that holds entry n of the full one (N odd),
// and the entry made from it; Im X[0] is ignored
__device__ __forceinline__ int odd_bin(int n, int N) { return 2 * n > N ? N - n : n; }
__device__ __forceinline__ c32 odd_full(int n, int N, c32 x) {
  const float y = 2 * n > N ? -x.y : x.y;
  return {x.x, n == 0 ? 0.0f : y};
}

// element n of transform b for the modes that need no twiddle, before the
// conjugation of the inverse
__device__ __forceinline__ c32 fs_input(const FsArgs& a, int64_t b, int n) {
  if (a.mode == FS_ODD_R2C) return {reinterpret_cast<const float*>(a.in)[b * a.ibs + n], 0.0f};
  if (a.mode == FS_ODD_C2R) return odd_full(n, a.N, a.in[b * a.ibs + odd_bin(n, a.N)]);
  return a.in[b * a.ibs + n];
}

// PAIR: two real columns a transform, 2b and 2b + 1, as the real and imaginary part
// (the last of an odd number of them alone).  With *wide one column's values could
// overflow into the other's: the block then takes 2b alone and, in a second turn
// (half = 1, results between the kernels at transform batch + b), 2b + 1.
__device__ __forceinline__ bool pair_second(const FsPair& p, int64_t b, int half) {
  return half == 0 && 2 * b + 1 < p.ncol;
}

// *p.wide by a vector load, which is waited for with the tile's own
__device__ __forceinline__ int pair_wide(const FsPair& p) {
  int lane0 = 0;
  asm volatile("" : "+v"(lane0));
  return p.wide[lane0] != 0 ? 1 : 0;
}

// element n of the pair's spectrum, A + i B, from its bins in the two columns
__device__ __forceinline__ c32 pair_full(int n, int N, c32 A, c32 B, bool two) {
  A = odd_full(n, N, A);
  B = two ? odd_full(n, N, B) : c32{0.0f, 0.0f};
  return {A.x - B.y, A.y + B.x};
}

// element k of the pair's columns
__device__ __forceinline__ void pair_output(const FsArgs& a, int64_t col, bool two, int k, c32 v) {
  float* out = reinterpret_cast<float*>(a.out) + col * a.obs + k;
  out[0] = v.x * a.scale;
  if (two) out[a.obs] = -v.y * a.scale;
}

// element k of transform b, scaled and (inverse) conjugated
__device__ __forceinline__ void fs_output(const FsArgs& a, int64_t b, int k, c32 v) {
  v = {v.x * a.scale, (a.inverse ? -v.y : v.y) * a.scale};
  if (a.mode == FS_ODD_C2R) {
    reinterpret_cast<float*>(a.out)[b * a.obs + k] = v.x;
  } else if (a.mode != FS_ODD_R2C || 2 * k < a.N) {
    a.out[b * a.obs + k] = v;
  }
}

// The unit of this block, of n units in all, such that each of the eight XCDs
// (blocks are dealt to them round-robin) takes one contiguous range of them;
// -1 for a block without one.  Neighbouring tiles share the cache lines at their
// edges (TC-element runs on rows that start anywhere) and so one XCD's L2: Nf =
// 10^6, 129 rates: fs_rows 370 -> 313 us, fs_cols 341 -> 329; 21609 x 234 rows
// 50 -> 48, columns unchanged.
__device__ __forceinline__ int64_t xcd_block(int64_t n) {
  const int64_t per = (n + 7) / 8;
  const int64_t u = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  return (blockIdx.x >> 3) < per && u < n ? u : -1;
}

// columns: block = (batch b, columns n2 in [c0, c0 + TC)); TC is a power of two.
// Thread: column c of the block, rows n0 + i dn; a transform's elements are within
// 2^23 bytes, so one base and 32-bit offsets reach them.  Loads past the edges
// take the last row or column and are not stored.
template <int TH, bool PAIR>
__device__ __forceinline__ void fs_cols_tile(const FsArgs& a, FsPairOf<PAIR> p, c32* lds, int64_t b, int c0, int half,
                                             int wide) {
  c32* buf = lds;
  // W_N^{n2 dr i}: with W_N^{n2 n0} of its own, a thread's four-step twiddles
  c32* step = lds + FS_PER * TH;
  c32* tw = step + 16 * FS_PER;
  const int TC = a.T;
  const int lgT = __ffs(TC) - 1;
  const int c = static_cast<int>(threadIdx.x) & (TC - 1), r0 = static_cast<int>(threadIdx.x) >> lgT;
  const int dr = TH >> lgT;
  const int col = min(c0 + c, a.N2 - 1);
  // all loads issued before the first LDS store
  c32 v[FS_PER];
  if constexpr (PAIR) {
    const bool two = pair_second(p, b, half);  // uniform
    const c32* A = a.in + (2 * b + half) * a.ibs;
    const c32* B = A + (two ? a.ibs : 0);
    c32 w[FS_PER];
#pragma unroll
    for (int i = 0; i < FS_PER; ++i) {
      if (i * dr < a.N1) {
        const uint32_t k = 8u * static_cast<uint32_t>(odd_bin(col + min(r0 + i * dr, a.N1 - 1) * a.N2, a.N));
        v[i] = at_byte(A, k);
        w[i] = at_byte(B, k);
      }
    }
#pragma unroll
    for (int i = 0; i < FS_PER; ++i)
      if (i * dr < a.N1)
        v[i] = pair_full(col + min(r0 + i * dr, a.N1 - 1) * a.N2, a.N, v[i], w[i], two && wide == 0);
  } else if (a.mode == FS_C2R) {
    const c32* X = a.in + b * a.ibs;
    const c32* Xe = X + a.N;
    c32 w[FS_PER];
#pragma unroll
    for (int i = 0; i < FS_PER; ++i) {
      if (i * dr < a.N1) {  // uniform
        const uint32_t k = 8u * static_cast<uint32_t>(col + min(r0 + i * dr, a.N1 - 1) * a.N2);
        v[i] = at_byte(X, k);
        w[i] = at_byte(X, 8u * static_cast<uint32_t>(a.N) - k);  // X[N] for k = 0
      }
    }
    const c32 w0 = cis_nh(-static_cast<double>(c0 + c + r0 * a.N2), 0.5 * a.h);
#pragma unroll
    for (int i = 0; i < FS_PER; ++i)
      if (i * dr < a.N1) v[i] = c2r_pack(c0 + c + r0 + i, v[i], w[i], cmul(w0, a.half[i]));
  } else if (a.mode == FS_C2C) {
    const c32* x = a.in + b * a.ibs;
#pragma unroll
    for (int i = 0; i < FS_PER; ++i)
      if (i * dr < a.N1)
        v[i] = at_byte(x, 8u * static_cast<uint32_t>(col + min(r0 + i * dr, a.N1 - 1) * a.N2));
  } else {
#pragma unroll
    for (int i = 0; i < FS_PER; ++i)
      if (i * dr < a.N1) v[i] = fs_input(a, b, col + min(r0 + i * dr, a.N1 - 1) * a.N2);
  }
  for (int i = threadIdx.x; i < a.ntw; i += TH) tw[i] = a.tw[i];
  if (static_cast<int>(threadIdx.x) < TC * FS_PER)
    step[threadIdx.x] = cis_nh(-static_cast<double>((c0 + c) * dr) * static_cast<double>(r0), a.h);
  const float sg = a.inverse ? -1.0f : 1.0f;
#pragma unroll
  for (int i = 0; i < FS_PER; ++i)  // element n of column c at n * TC + c; rows past N1 land behind the last one
    if (i * dr < a.N1) buf[static_cast<int>(threadIdx.x) + i * TH] = {v[i].x, sg * v[i].y};
  __syncthreads();
  fs_dft<TH>(buf, tw, a, a.N1);
  if (c0 + c >= a.N2) return;
  c32* dst = a.out + (PAIR ? b + half * a.batch : b) * a.N + c0;
  int k0 = r0;
  asm volatile("" : "+v"(k0));  // keeps the store indices from being computed before the passes
  const c32 w0 = cis_nh(-static_cast<double>((c0 + c) * k0), a.h);
  const uint32_t o0 = 8u * static_cast<uint32_t>(c + k0 * a.N2), od = 8u * static_cast<uint32_t>(dr * a.N2);
  const uint32_t l0 = 8u * static_cast<uint32_t>(k0 * TC + c);
#pragma unroll
  for (int i = 0; i < FS_PER; ++i)
    if (k0 + i * dr < a.N1)
      at_byte(dst, o0 + static_cast<uint32_t>(i) * od) = cmul(at_byte(buf, l0 + 8u * TH * i), cmul(w0, step[i * TC + c]));
}

template <int TH, bool PAIR>
__global__ __launch_bounds__(TH, 8) void fs_cols(FsArgs a, FsPairOf<PAIR> p) {
  extern __shared__ __align__(16) c32 lds[];  // FS_PER TH elements, the steps, the passes' twiddles
  const int tiles = (a.N2 + a.T - 1) / a.T;
  const int64_t blk = xcd_block(tiles * a.batch);
  if (blk < 0) return;
  const int64_t b = blk / tiles;
  const int c0 = static_cast<int>(blk % tiles) * a.T;
  if constexpr (PAIR) {
    const int wide = pair_wide(p);
    fs_cols_tile<TH, true>(a, p, lds, b, c0, 0, wide);
    if (!pair_second(p, b, 0) || __builtin_amdgcn_readfirstlane(wide) == 0) return;  // uniform
    __syncthreads();
    fs_cols_tile<TH, true>(a, p, lds, b, c0, 1, wide);  // a loop over both turns would spill
  } else {
    fs_cols_tile<TH, false>(a, p, lds, b, c0, 0, 0);
  }
}

// rows: block = (batch b, rows k1 in [r0, r0 + TR)); TR is a power of two.  Rows are
// interleaved as in fs_cols (element n of row c at n * TR + c), which keeps the
// passes' LDS accesses as conflict-free as fs_cols's.
template <int TH, bool PAIR>
__device__ __forceinline__ void fs_rows_tile(const FsArgs& a, FsPairOf<PAIR> p, c32* lds, int64_t b, int r0, int half,
                                             int wide) {
  c32* buf = lds;
  const c32* tw = lds + FS_PER * TH;
  const int TR = a.T;
  const int lgT = __ffs(TR) - 1;
  const int c = static_cast<int>(threadIdx.x) & (TR - 1), n0 = static_cast<int>(threadIdx.x) >> lgT;
  const int dn = TH >> lgT;
  {
    const c32* src = a.in + (PAIR ? b + half * a.batch : b) * a.N;
    const int row = min(r0 + c, a.N1 - 1) * a.N2;
    c32 v[FS_PER];
#pragma unroll
    for (int i = 0; i < FS_PER; ++i)
      if (i * dn < a.N2) v[i] = at_byte(src, 8u * static_cast<uint32_t>(row + min(n0 + i * dn, a.N2 - 1)));
#pragma unroll
    for (int i = 0; i < FS_PER; ++i)
      if (i * dn < a.N2) buf[static_cast<int>(threadIdx.x) + i * TH] = v[i];
  }
  __syncthreads();
  fs_dft<TH>(buf, tw, a, a.N2);
  if (r0 + c >= a.N1) return;
  int k2 = n0;
  asm volatile("" : "+v"(k2));  // keeps the store indices from being computed before the passes
  const uint32_t l0 = 8u * static_cast<uint32_t>(k2 * TR + c);
  if constexpr (PAIR) {
    const bool two = wide == 0 && pair_second(p, b, half);
#pragma unroll
    for (int i = 0; i < FS_PER; ++i)
      if (k2 + i * dn < a.N2)
        pair_output(a, 2 * b + half, two, r0 + c + (k2 + i * dn) * a.N1, at_byte(buf, l0 + 8u * TH * i));
  } else if (a.mode == FS_C2C || a.mode == FS_C2R) {
    const float sx = a.scale, sy = a.inverse ? -a.scale : a.scale;
    c32* dst = a.out + b * a.obs + r0;
    const uint32_t o0 = 8u * static_cast<uint32_t>(c + k2 * a.N1), od = 8u * static_cast<uint32_t>(dn * a.N1);
#pragma unroll
    for (int i = 0; i < FS_PER; ++i)
      if (k2 + i * dn < a.N2) {
        const c32 z = at_byte(buf, l0 + 8u * TH * i);
        at_byte(dst, o0 + static_cast<uint32_t>(i) * od) = {z.x * sx, z.y * sy};
      }
  } else {
#pragma unroll
    for (int i = 0; i < FS_PER; ++i)
      if (k2 + i * dn < a.N2)
        fs_output(a, b, r0 + c + (k2 + i * dn) * a.N1, at_byte(buf, l0 + 8u * TH * i));
  }
}

template <int TH, bool PAIR>
__global__ __launch_bounds__(TH, 8) void fs_rows(FsArgs a, FsPairOf<PAIR> p) {
  extern __shared__ __align__(16) c32 lds[];  // FS_PER TH elements, the passes' twiddles
  // (their loads are under way during the divisions below)
  for (int i = threadIdx.x; i < a.ntw; i += TH) lds[FS_PER * TH + i] = a.tw[i];
  const int tiles = (a.N1 + a.T - 1) / a.T;
  const int64_t blk = xcd_block(tiles * a.batch);
  if (blk < 0) return;
  const int64_t b = blk / tiles;
  const int r0 = static_cast<int>(blk % tiles) * a.T;
  if constexpr (PAIR) {
    const int wide = pair_wide(p);
    fs_rows_tile<TH, true>(a, p, lds, b, r0, 0, wide);
    if (!pair_second(p, b, 0) || __builtin_amdgcn_readfirstlane(wide) == 0) return;  // uniform
    __syncthreads();
    fs_rows_tile<TH, true>(a, p, lds, b, r0, 1, wide);  // a loop over both turns would spill
  } else {
    fs_rows_tile<TH, false>(a, p, lds, b, r0, 0, 0);
  }
}

// whole transforms: block = transforms [T blockIdx, T blockIdx + T), element n of
// transform c at n * T + c; LDS: N * T elements, then the twiddles
template <bool PAIR>
__device__ __forceinline__ void fs_one_tile(const FsArgs& a, FsPairOf<PAIR> p, c32* lds, int half, int wide) {
  constexpr int TH = FS_ONE_TH;
  c32* buf = lds;
  c32* tw = lds + a.N * a.T;
  for (int i = threadIdx.x; i < a.ntw; i += TH) tw[i] = a.tw[i];
  const int64_t b0 = static_cast<int64_t>(blockIdx.x) * a.T;
  const int nt = static_cast<int>(min(static_cast<int64_t>(a.T), a.batch - b0));
  const int E = a.N * nt;
  const FsDiv dN = fs_div(a.N);
  {
    // loads past the last element take it again; one branch on the mode around them
    // all, so that they are in flight together
    c32 v[FS_PER], w[FS_PER];
    auto each = [&](auto&& f) {
#pragma unroll
      for (int i = 0; i < FS_PER; ++i) {
        const int e = min(static_cast<int>(threadIdx.x) + i * TH, E - 1);
        const int c = fs_quo(e, dN), n = e - c * a.N;
        f(i, b0 + c, n);
      }
    };
    if constexpr (PAIR) {
      each([&](int i, int64_t u, int n) {
        const c32* A = a.in + min(2 * u + half, p.ncol - 1) * a.ibs + odd_bin(n, a.N);
        v[i] = A[0];
        w[i] = A[pair_second(p, u, half) ? a.ibs : 0];
      });
      each([&](int i, int64_t u, int n) {
        v[i] = pair_full(n, a.N, v[i], w[i], wide == 0 && pair_second(p, u, half));
      });
    } else if (a.mode == FS_C2R) {
      each([&](int i, int64_t b, int n) {
        const c32* X = a.in + b * a.ibs;
        v[i] = X[n];
        w[i] = X[a.N - n];
      });
      each([&](int i, int64_t, int n) {
        v[i] = c2r_pack(n, v[i], w[i], cis_nh(-static_cast<double>(n), 0.5 * a.h));
      });
    } else if (a.mode == FS_ODD_C2R) {
      each([&](int i, int64_t b, int n) { v[i] = a.in[b * a.ibs + odd_bin(n, a.N)]; });
      each([&](int i, int64_t, int n) { v[i] = odd_full(n, a.N, v[i]); });
    } else if (a.mode == FS_ODD_R2C) {
      each([&](int i, int64_t b, int n) {
        v[i] = {reinterpret_cast<const float*>(a.in)[b * a.ibs + n], 0.0f};
      });
    } else {
      each([&](int i, int64_t b, int n) { v[i] = a.in[b * a.ibs + n]; });
    }
#pragma unroll
    for (int i = 0; i < FS_PER; ++i) {
      const int e = static_cast<int>(threadIdx.x) + i * TH;
      const int c = fs_quo(e, dN), n = e - c * a.N;
      if (e < E) buf[n * a.T + c] = {v[i].x, a.inverse ? -v[i].y : v[i].y};
    }
  }
  __syncthreads();
  fs_dft<TH>(buf, tw, a, a.N);
  int tid = static_cast<int>(threadIdx.x);
  asm volatile("" : "+v"(tid));
  if (!PAIR && a.mode == FS_R2C) {
    // X[k] = E + W_{2N}^k O, X[N-k] = conj(E - W_{2N}^k O), E = (Z[k] + conj Z[N-k])/2,
    // O = (Z[k] - conj Z[N-k])/(2i)
    const int half = a.N / 2 + 1;
    const FsDiv dH = fs_div(half);
    for (int e = tid; e < half * nt; e += TH) {
      const int c = fs_quo(e, dH), k = e - c * half;
      c32* x = a.out + (b0 + c) * a.obs;
      const c32 z = buf[k * a.T + c];
      if (k == 0) {
        x[0] = {z.x + z.y, 0.0f};
        x[a.N] = {z.x - z.y, 0.0f};
      } else {
        const c32 y = buf[(a.N - k) * a.T + c];
        const c32 Ev = {0.5f * (z.x + y.x), 0.5f * (z.y - y.y)};
        const c32 O = {0.5f * (z.y + y.y), -0.5f * (z.x - y.x)};
        const c32 WO = cmul(cis_nh(-static_cast<double>(k), 0.5 * a.h), O);
        x[k] = cadd(Ev, WO);
        if (2 * k != a.N) x[a.N - k] = {Ev.x - WO.x, -(Ev.y - WO.y)};
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < FS_PER; ++i) {
    const int e = tid + i * TH;
    const int c = fs_quo(e, dN), k = e - c * a.N;
    if (e < E) {
      if constexpr (PAIR) {
        const int64_t u = b0 + c;
        if (2 * u + half < p.ncol)
          pair_output(a, 2 * u + half, wide == 0 && pair_second(p, u, half), k, buf[k * a.T + c]);
      } else {
        fs_output(a, b0 + c, k, buf[k * a.T + c]);
      }
    }
  }
}

template <bool PAIR>
__global__ __launch_bounds__(FS_ONE_TH, 4) void fs_one(FsArgs a, FsPairOf<PAIR> p) {
  extern __shared__ __align__(16) c32 lds[];
  if constexpr (PAIR) {
    const int wide = pair_wide(p);
    fs_one_tile<true>(a, p, lds, 0, wide);
    if (__builtin_amdgcn_readfirstlane(wide) == 0) return;  // uniform
    __syncthreads();
    fs_one_tile<true>(a, p, lds, 1, wide);
  } else {
    fs_one_tile<false>(a, p, lds, 0, 0);
  }
}

static bool fs_has(const FftPlan* p) { return !p->rad0.empty() || p->N1 > 0; }

static void fs_passes(FsArgs* a, const std::vector<int>& rad, const c32* tw) {
  a->np = static_cast<int>(rad.size());
  int Ns = 1;
  a->ntw = 0;
  for (int i = 0; i < a->np; ++i) {
    a->rad[i] = rad[i];
    if (Ns > 1) a->ntw += (rad[i] - 1) * Ns;
    Ns *= rad[i];
  }
  a->tw = tw;
}

// `batch` transforms of plan p in mode `mode`; the result is multiplied by
// scale.  s0: scratch of N * batch elements (four-step only).  wide: two real columns
// a transform (FS_ODD_C2R; batch and s0 count the columns)
static int fs_run(const FftPlan* p, int mode, const void* in, int64_t ibs, void* out, int64_t obs, int64_t batch,
                  bool inverse, double scale, c32* s0, hipStream_t st, const int64_t* wide = nullptr) {
  FsArgs a;
  const FsPair pr = {batch, wide};
  if (wide != nullptr) batch = (batch + 1) / 2;
  a.N = static_cast<int>(p->N);
  a.N1 = p->N1;
  a.N2 = p->N2;
  a.inverse = inverse ? 1 : 0;
  a.batch = batch;
  a.h = 1.0 / static_cast<double>(p->N);
  const double bytes = 16.0 * static_cast<double>(p->N) * static_cast<double>(batch);
  if (!p->rad0.empty()) {
    a.in = static_cast<const c32*>(in);
    a.ibs = ibs;
    a.out = static_cast<c32*>(out);
    a.obs = obs;
    a.mode = mode;
    a.scale = static_cast<float>(scale);
    // as many transforms a block as fit, but blocks for every CU first
    int T = std::min<int>(16, pow2_floor(FS_ONE / p->N));
    while (T > 1 && batch / T < 512) T /= 2;
    a.T = T;
    fs_passes(&a, p->rad0, p->tw0);
    const size_t lds = (static_cast<size_t>(p->N) * T + a.ntw) * sizeof(c32);
    ProfScope ps(st, "fft_fs_one", bytes);
    const unsigned grid = static_cast<unsigned>((batch + T - 1) / T);
    if (wide != nullptr) fs_one<true><<<grid, FS_ONE_TH, lds, st>>>(a, pr);
    else fs_one<false><<<grid, FS_ONE_TH, lds, st>>>(a, {});
    ZDT_CHECK_LAUNCH("fs_one");
    return ZDT_OK;
  }
  {
    a.in = static_cast<const c32*>(in);
    a.ibs = ibs;
    a.out = s0;
    a.obs = p->N;
    a.mode = mode;
    a.T = p->TC;
    a.scale = 1.0f;
    const int64_t grid = ((p->N2 + p->TC - 1) / p->TC * batch + 7) / 8 * 8;
    const int E = p->N1 * p->TC;
    // Threads for 8 elements each: the fewest that cover the block keep its passes'
    // wavefronts full and fit more blocks a CU; a grid of one round is better off
    // with more of them.  Columns of 147 x 16 (21609 x 234, 205 rates): 1024 threads
    // 125 us, 512 73, 320 58; of 125 x 16 in 200 blocks: 320 20, 512 16; of 576 x 8
    // (1179648, 100 rates), where wavefronts a CU matter more: 640 366, 1024 305.
    const int th = E > 512 * FS_PER ? 1024 : E > 320 * FS_PER || grid < 512 ? 512 : 320;
    for (int i = 0; i < FS_PER; ++i) {
      const double x = 3.14159265358979323846 * i * (th / p->TC) / p->N1;
      a.half[i] = {static_cast<float>(std::cos(x)), static_cast<float>(-std::sin(x))};
    }
    fs_passes(&a, p->rad1, p->tw1);
    ProfScope ps(st, mode == FS_C2R ? "fft_fs_cols_c2r" : "fft_fs_cols", bytes);
    const size_t lds = (FS_PER * th + 16 * FS_PER + a.ntw) * sizeof(c32);
    const unsigned g = static_cast<unsigned>(grid);
    if (wide != nullptr) {
      const auto kern = th == 320 ? fs_cols<320, true> : th == 512 ? fs_cols<512, true> : fs_cols<1024, true>;
      kern<<<g, th, lds, st>>>(a, pr);
    } else {
      const auto kern = th == 320 ? fs_cols<320, false> : th == 512 ? fs_cols<512, false> : fs_cols<1024, false>;
      kern<<<g, th, lds, st>>>(a, {});
    }
    ZDT_CHECK_LAUNCH("fs_cols");
  }
  {
    a.in = s0;
    a.ibs = p->N;
    a.out = static_cast<c32*>(out);
    a.obs = obs;
    a.T = p->TR;
    a.scale = static_cast<float>(scale);
    fs_passes(&a, p->rad2, p->tw2);
    const int64_t grid = ((p->N1 + p->TR - 1) / p->TR * batch + 7) / 8 * 8;
    ProfScope ps(st, "fft_fs_rows", bytes);
    const int th = p->N2 * p->TR > 512 * FS_PER ? 1024 : 512;
    const size_t lds = (FS_PER * th + a.ntw) * sizeof(c32);
    const unsigned g = static_cast<unsigned>(grid);
    if (wide != nullptr) {
      const auto kern = th == 512 ? fs_rows<512, true> : fs_rows<1024, true>;
      kern<<<g, th, lds, st>>>(a, pr);
    } else {
      const auto kern = th == 512 ? fs_rows<512, false> : fs_rows<1024, false>;
      kern<<<g, th, lds, st>>>(a, {});
    }
    ZDT_CHECK_LAUNCH("fs_rows");
  }
  return ZDT_OK;
}

// Radices of an LDS transform of length n with the fewest passes (fewest large
// ones among those): composite and power-of-two radices up to maxr, primes up to 13.
// False if n has another prime factor.
static bool fs_radices(int64_t n, int maxr, std::vector<int>* best) {
  best->clear();
  if (n == 1) return true;
  bool found = false;
  for (int r : {16, 15, 14, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2}) {
    const bool prime = r == 2 || r == 3 || r == 5 || r == 7 || r == 11 || r == 13;
    if (n % r != 0 || (!prime && r > maxr)) continue;
    std::vector<int> sub;
    if (!fs_radices(n / r, std::min(maxr, r), &sub)) continue;  // non-increasing
    if (!sub.empty() && sub[0] > r) continue;
    if (!found || sub.size() + 1 <= best->size()) {  // later candidates start smaller
      best->assign(1, r);
      best->insert(best->end(), sub.begin(), sub.end());
      found = true;
    }
  }
  return found;
}

// Chooses the LDS form of an FP32 plan (neither if none applies): one kernel, or
// the four-step split whose column and row blocks both move the longest
// contiguous runs and, among those, takes the fewest passes.
static void fs_choose(FftPlan* p, int maxr) {
  p->N1 = 0;
  const int64_t N = p->N;
  if (p->dbl || N < 2) return;
  if (N <= FS_ONE) {
    if (!fs_radices(N, maxr, &p->rad0) || static_cast<int>(p->rad0.size()) > FS_MAXP) p->rad0.clear();
    return;
  }
  if (N > (int64_t{1} << 20)) return;
  int best = -1;
  for (int64_t n1 = 2; n1 <= 1024; ++n1) {
    if (N % n1 != 0) continue;
    const int64_t n2 = N / n1;
    if (n2 < 2 || n2 > 2048) continue;
    std::vector<int> r1, r2;
    if (!fs_radices(n1, maxr, &r1) || !fs_radices(n2, maxr, &r2)) continue;
    if (static_cast<int>(r1.size()) > FS_MAXP || static_cast<int>(r2.size()) > FS_MAXP) continue;
    const int tc = std::min(16, pow2_floor(FS_E / n1));
    const int tr = std::min(16, pow2_floor(FS_E / n2));
    const int score = (std::min(tc, tr) * 100 + tc) * 32 + 31 - static_cast<int>(r1.size() + r2.size());
    if (score > best) {
      best = score;
      p->N1 = static_cast<int>(n1);
      p->N2 = static_cast<int>(n2);
      p->TC = tc;
      p->TR = tr;
      p->rad1 = r1;
      p->rad2 = r2;
    }
  }
}

// Gain of a radix: the mean over its outputs of Re sum_j M~[k][j] conj(M[k][j]) / R - 1
// for the matrix M~ that its constants give once they are rounded to 32 bits.  The
// passes repeat the same few constants, so these add up (10^6 channels: 1.6e-7
// over both transforms) where the errors of a table's many entries average out.
static constexpr double FS_GAIN[17] = {0, 0,        0,       -6.0e-9, 0,        8.6e-9, -1.05e-8, -4.6e-9, -4.3e-9,
                                       -1.57e-8, 1.4e-8, -3.3e-9, -1.05e-8, 0.6e-9, -7.3e-9,  7.0e-9,  -1.36e-8};
// and of the two factors of a four-step twiddle (cis_nh)
static constexpr double FS_GAIN_STEP = 1.5e-8;

// the passes' twiddles W_{Ns R}^{r k} (r = 1 .. R-1, k < Ns) of every pass but the
// first, in order, scaled so that the passes' gains and `gain` cancel: gain of a tone
// over both transforms, 35 lengths from 2000 to 1.2 million, rms 1.1e-7 -> 1.6e-8.
// (Double sines: 4096 entries in 0.1 to 0.4 ms on the host, against 0.7 to 0.8 from
// 80-bit ones; unscaled, all entries of lengths up to 4096 round to the same 32 bits.)
static std::vector<c32> fs_twiddles(const std::vector<int>& rad, double gain) {
  std::vector<c32> t;
  int64_t Ns = 1;
  for (int R : rad) {
    gain += FS_GAIN[R];
    if (Ns > 1) {
      // (those of r = 0 and k = 0 are 1, so that the mean, which no constant touches, is exact)
      const double unit = 1.0 - gain * R * Ns / ((R - 1) * (Ns - 1));
      for (int r = 1; r < R; ++r)
        for (int64_t k = 0; k < Ns; ++k) {
          const int64_t n = Ns * R, m = r * k;  // m < n
          const double x = 6.283185307179586 * static_cast<double>(m) / static_cast<double>(n);
          double c = std::cos(x), sn = -std::sin(x);
          if (4 * m == n || 4 * m == 3 * n) c = 0.0;
          if (2 * m == n) sn = 0.0;
          t.push_back(k == 0 ? c32{1.0f, 0.0f} : c32{static_cast<float>(unit * c), static_cast<float>(unit * sn)});
        }
      gain = 0.0;
    }
    Ns *= R;
  }
  return t;
}

// ---------------------------------------------------------------- plans

bool fft_factorize(int64_t N, std::vector<int>* radices, int maxr) {
  radices->clear();
  if (N < 1) return false;
  int64_t n = N;
  for (int r : {16, 8, 4, 2, 3, 5, 7, 11, 13}) {
    if ((r & (r - 1)) == 0 && r > maxr) continue;  // power-of-two radices above the cap
    while (n % r == 0) {
      radices->push_back(r);
      n /= r;
    }
  }
  return n == 1;
}

namespace {
struct PlanKey {
  int device;
  int64_t N;
  bool dbl;
  int maxr;
  bool operator<(const PlanKey& o) const {
    return std::tie(device, N, dbl, maxr) < std::tie(o.device, o.N, o.dbl, o.maxr);
  }
};
std::mutex g_plan_mu;
std::map<PlanKey, FftPlan*> g_plans;
}  // namespace

int fft_plan_get(int64_t N, bool dbl, const FftPlan** out, int maxr) {
  std::vector<int> radices;
  if (maxr != 16 && maxr != 8 && maxr != 4) return fail(ZDT_EINVAL, "FFT radix cap must be 4, 8 or 16");
  if (!fft_factorize(N, &radices, maxr))
    return fail(ZDT_ENOTSUP, "FFT length %lld has a prime factor outside {2,3,5,7,11,13}",
                static_cast<long long>(N));
  int dev = 0;
  ZDT_TRY_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_plan_mu);
  PlanKey key{dev, N, dbl, maxr};
  auto it = g_plans.find(key);
  if (it != g_plans.end()) {
    *out = it->second;
    return ZDT_OK;
  }
  FftPlan* p = new FftPlan();
  p->N = N;
  p->dbl = dbl;
  p->radices = radices;
  // twiddle table W_N^m = exp(-2 pi i m / N), m < N, from an exact reduction
  const size_t esz = dbl ? sizeof(c64) : sizeof(c32);
  std::vector<unsigned char> host(static_cast<size_t>(N) * esz);
  for (int64_t m = 0; m < N; ++m) {
    // angle = 2 pi m/N; use the symmetric quarter to keep cos/sin exact at
    // multiples of pi/2
    const long double a = 2.0L * 3.14159265358979323846264338327950288L * static_cast<long double>(m) /
                          static_cast<long double>(N);
    double c = static_cast<double>(cosl(a));
    double s = -static_cast<double>(sinl(a));
    if (4 * m == N || 4 * m == 3 * N) c = 0.0;
    if (2 * m == N) s = 0.0;
    if (dbl) {
      reinterpret_cast<c64*>(host.data())[m] = {c, s};
    } else {
      reinterpret_cast<c32*>(host.data())[m] = {static_cast<float>(c), static_cast<float>(s)};
    }
  }
  hipError_t e = hipMalloc(&p->tw, host.size());
  if (e != hipSuccess) {
    delete p;
    return fail(ZDT_ENOMEM, "hipMalloc of FFT twiddles (%zu bytes) failed", host.size());
  }
  e = hipMemcpy(p->tw, host.data(), host.size(), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    (void)hipFree(p->tw);
    delete p;
    return hip_fail(e, "hipMemcpy(twiddles)");
  }
  fs_choose(p, maxr);
  {
    // one allocation for the passes' twiddles of whichever forms the plan has
    const std::vector<c32> t0 = fs_twiddles(p->rad0, 0.0), t1 = fs_twiddles(p->rad1, FS_GAIN_STEP),
                           t2 = fs_twiddles(p->rad2, 0.0);
    std::vector<c32> all(t0);
    all.insert(all.end(), t1.begin(), t1.end());
    all.insert(all.end(), t2.begin(), t2.end());
    if (!all.empty()) {
      c32* d = nullptr;
      e = hipMalloc(&d, all.size() * sizeof(c32));
      if (e != hipSuccess) {
        (void)hipFree(p->tw);
        delete p;
        return fail(ZDT_ENOMEM, "hipMalloc of FFT twiddles failed");
      }
      e = hipMemcpy(d, all.data(), all.size() * sizeof(c32), hipMemcpyHostToDevice);
      if (e != hipSuccess) {
        (void)hipFree(d);
        (void)hipFree(p->tw);
        delete p;
        return hip_fail(e, "hipMemcpy(twiddles)");
      }
      p->tw0 = d;
      p->tw1 = d + t0.size();
      p->tw2 = d + t0.size() + t1.size();
    }
  }
  g_plans[key] = p;
  *out = p;
  return ZDT_OK;
}

template <typename T>
static int c2c_impl(const FftPlan* p, const void* in, int64_t ies, int64_t ibs, void* out, int64_t oes,
                    int64_t obs, int64_t batch, bool inverse, double scale, void* s0, void* s1,
                    hipStream_t st) {
  const int np = static_cast<int>(p->radices.size());
  const int64_t N = p->N;
  const cplx<T>* tw = static_cast<const cplx<T>*>(p->tw);
  if constexpr (std::is_same<T, float>::value) {
    if (fs_has(p) && ies == 1 && oes == 1)
      return fs_run(p, FS_C2C, in, ibs, out, obs, batch, inverse, scale, static_cast<c32*>(s0), st);
  }
  if (N == 1) {
    // the length-1 DFT is the identity (times scale)
    scale_copy<T><<<grid_for(batch, 256), 256, 0, st>>>(static_cast<const cplx<T>*>(in), ibs,
                                                        static_cast<cplx<T>*>(out), obs, batch,
                                                        static_cast<T>(scale));
    ZDT_CHECK_LAUNCH("scale_copy");
    return ZDT_OK;
  }
  int64_t Ns = 1;
  const void* src = in;
  int64_t ses = ies, sbs = ibs;
  for (int pi = 0; pi < np; ++pi) {
    const int R = p->radices[pi];
    const bool last = (pi == np - 1);
    void* dst = last ? out : ((pi & 1) ? s1 : s0);
    const int64_t des = last ? oes : 1;
    const int64_t dbs = last ? obs : N;
    PassArgs a;
    a.N = N;
    a.NR = N / R;
    a.Ns = Ns;
    a.twstep = N / (Ns * R);
    a.ies = ses;
    a.ibs = sbs;
    a.oes = des;
    a.obs = dbs;
    a.batch = batch;
    a.scale = last ? scale : 1.0;
    a.inverse = inverse ? 1 : 0;
    // consecutive lanes along the contiguous index
    a.jmajor = (ses == 1 || batch == 1) ? 1 : 0;
    ZDT_TRY(launch_pass<T>(R, static_cast<const cplx<T>*>(src), static_cast<cplx<T>*>(dst), tw, a, st));
    Ns *= R;
    src = dst;
    ses = des;
    sbs = dbs;
  }
  return ZDT_OK;
}

int fft_c2c(const FftPlan* p, const void* in, int64_t ies, int64_t ibs, void* out, int64_t oes,
            int64_t obs, int64_t batch, bool inverse, double scale, void* s0, void* s1, hipStream_t st) {
  if (p->dbl)
    return c2c_impl<double>(p, in, ies, ibs, out, oes, obs, batch, inverse, scale, s0, s1, st);
  return c2c_impl<float>(p, in, ies, ibs, out, oes, obs, batch, inverse, scale, s0, s1, st);
}

// ---------------------------------------------------------------- real transforms

// r2c post-processing for even N = 2M.  Z = FFT_M(x[2n] + i x[2n+1]).
// X[k] = (Z[k] + conj Z[M-k])/2 - i W_N^k (Z[k] - conj Z[M-k])/2, k in [0, M].
__global__ __launch_bounds__(256) void r2c_post(const c32* __restrict__ Z, c32* __restrict__ X,
                                                const c32* __restrict__ twN, int64_t M, int64_t ldx,
                                                int64_t batch) {
  const int64_t half = M / 2 + 1;  // k in [0, M/2]
  const int64_t total = half * batch;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < total;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t k = g % half, b = g / half;
    const c32* z = Z + b * M;
    c32* x = X + b * ldx;
    if (k == 0) {
      const c32 z0 = z[0];
      x[0] = {z0.x + z0.y, 0.0f};
      x[M] = {z0.x - z0.y, 0.0f};
      continue;
    }
    const int64_t km = M - k;
    const c32 a = z[k], bb = z[km];
    {
      // E = (a + conj bb)/2, O = (a - conj bb)/(2i)
      const c32 E = {0.5f * (a.x + bb.x), 0.5f * (a.y - bb.y)};
      const c32 O = {0.5f * (a.y + bb.y), -0.5f * (a.x - bb.x)};
      x[k] = cadd(E, cmul(twN[k], O));
    }
    if (km != k) {
      const c32 E = {0.5f * (bb.x + a.x), 0.5f * (bb.y - a.y)};
      const c32 O = {0.5f * (bb.y + a.y), -0.5f * (bb.x - a.x)};
      x[km] = cadd(E, cmul(twN[km], O));
    }
  }
}

// c2r pre-processing for even N = 2M.  The imaginary parts of X[0] and X[M]
// are ignored (the c2r convention of FFTW/cuFFT).  Z'[k] = (E + i O) * scale
// with E = (X[k] + conj X[M-k])/2, O = W_N^{-k} (X[k] - conj X[M-k])/2.
__global__ __launch_bounds__(256) void c2r_pre(const c32* __restrict__ X, c32* __restrict__ Z,
                                               const c32* __restrict__ twN, int64_t M, int64_t ldx,
                                               int64_t batch, float scale) {
  const int64_t half = M / 2 + 1;
  const int64_t total = half * batch;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < total;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t k = g % half, b = g / half;
    const c32* x = X + b * ldx;
    c32* z = Z + b * M;
    if (k == 0) {
      const float a = x[0].x, c = x[M].x;
      z[0] = {0.5f * (a + c) * scale, 0.5f * (a - c) * scale};
      continue;
    }
    const int64_t km = M - k;
    const c32 p = x[k], q = x[km];
    {
      const c32 E = {0.5f * (p.x + q.x), 0.5f * (p.y - q.y)};
      const c32 D = {0.5f * (p.x - q.x), 0.5f * (p.y + q.y)};
      const c32 O = cmulc(D, twN[k]);  // D * conj(W^k) = W^{-k} D
      z[k] = {(E.x - O.y) * scale, (E.y + O.x) * scale};
    }
    if (km != k) {
      const c32 E = {0.5f * (q.x + p.x), 0.5f * (q.y - p.y)};
      const c32 D = {0.5f * (q.x - p.x), 0.5f * (q.y + p.y)};
      const c32 O = cmulc(D, twN[km]);
      z[km] = {(E.x - O.y) * scale, (E.y + O.x) * scale};
    }
  }
}

// odd N helpers
__global__ __launch_bounds__(256) void real_to_complex(const float* __restrict__ in, int64_t ldi,
                                                       c32* __restrict__ out, int64_t N, int64_t batch) {
  const int64_t total = N * batch;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < total;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t n = g % N, b = g / N;
    out[b * N + n] = {in[b * ldi + n], 0.0f};
  }
}

__global__ __launch_bounds__(256) void copy_rows(const c32* __restrict__ in, int64_t ldi,
                                                 c32* __restrict__ out, int64_t ldo, int64_t rows,
                                                 int64_t batch) {
  const int64_t total = rows * batch;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < total;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t n = g % rows, b = g / rows;
    out[b * ldo + n] = in[b * ldi + n];
  }
}

// full Hermitian spectrum of length N (odd) from Nk = (N+1)/2 bins; Im X[0] ignored
__global__ __launch_bounds__(256) void hermitian_extend(const c32* __restrict__ X, int64_t ldx,
                                                        c32* __restrict__ full, int64_t N,
                                                        int64_t batch) {
  const int64_t total = N * batch;
  const int64_t Nk = N / 2 + 1;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < total;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t n = g % N, b = g / N;
    c32 v;
    if (n == 0) {
      v = {X[b * ldx].x, 0.0f};
    } else if (n < Nk) {
      v = X[b * ldx + n];
    } else {
      v = cconj(X[b * ldx + (N - n)]);
    }
    full[b * N + n] = v;
  }
}

__global__ __launch_bounds__(256) void complex_real_part(const c32* __restrict__ in, float* __restrict__ out,
                                                         int64_t ldo, int64_t N, int64_t batch) {
  const int64_t total = N * batch;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < total;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t n = g % N, b = g / N;
    out[b * ldo + n] = in[b * N + n].x;
  }
}

size_t fft_real_scratch_elems(int64_t N, int64_t batch) {
  const int64_t n = (N % 2 == 0) ? N / 2 : N;
  return static_cast<size_t>(n) * static_cast<size_t>(batch);
}

int fft_r2c(int64_t N, const float* in, int64_t ldi, c32* out, int64_t ldo, int64_t batch, void* s0,
            void* s1, void* s2, hipStream_t st, int maxr) {
  if (N % 2 == 0) {
    const int64_t M = N / 2;
    if (ldi % 2 != 0) return fail(ZDT_EINVAL, "r2c: column stride must be even for even N");
    const FftPlan *pM = nullptr, *pN = nullptr;
    ZDT_TRY(fft_plan_get(N, false, &pN, maxr));
    c32* Z = static_cast<c32*>(s2);
    if (M == 1) {
      // length-1 complex FFT of the packed pair is the pair itself
      ZDT_TRY_HIP(hipMemcpy2DAsync(Z, sizeof(c32), in, ldi * sizeof(float), sizeof(c32), batch,
                                   hipMemcpyDeviceToDevice, st));
    } else {
      ZDT_TRY(fft_plan_get(M, false, &pM, maxr));
      if (!pM->rad0.empty())  // the untangling in the same kernel
        return fs_run(pM, FS_R2C, in, ldi / 2, out, ldo, batch, false, 1.0, nullptr, st);
      ZDT_TRY(fft_c2c(pM, in, 1, ldi / 2, Z, 1, M, batch, false, 1.0, s0, s1, st));
    }
    ProfScope ps(st, "r2c_post", 16.0 * static_cast<double>(M * batch));
    r2c_post<<<grid_for((M / 2 + 1) * batch, 256), 256, 0, st>>>(Z, out, static_cast<const c32*>(pN->tw),
                                                                   M, ldo, batch);
    ZDT_CHECK_LAUNCH("r2c_post");
    return ZDT_OK;
  }
  const FftPlan* p = nullptr;
  ZDT_TRY(fft_plan_get(N, false, &p, maxr));
  if (fs_has(p)) return fs_run(p, FS_ODD_R2C, in, ldi, out, ldo, batch, false, 1.0, static_cast<c32*>(s0), st);
  c32* full = static_cast<c32*>(s2);
  real_to_complex<<<grid_for(N * batch, 256), 256, 0, st>>>(in, ldi, full, N, batch);
  ZDT_CHECK_LAUNCH("real_to_complex");
  // N odd and > 1: FFT into s0/s1 chain, final result into s0 region is not
  // allowed (scratch), so transform in place on `full`.
  ZDT_TRY(fft_c2c(p, full, 1, N, full, 1, N, batch, false, 1.0, s0, s1, st));
  copy_rows<<<grid_for((N / 2 + 1) * batch, 256), 256, 0, st>>>(full, N, out, ldo, N / 2 + 1, batch);
  ZDT_CHECK_LAUNCH("copy_rows");
  return ZDT_OK;
}

int fft_c2r(int64_t N, const c32* in, int64_t ldi, float* out, int64_t ldo, int64_t batch, double scale,
            void* s0, void* s1, void* s2, hipStream_t st, int maxr, const int64_t* wide) {
  if (N % 2 == 0) {
    const int64_t M = N / 2;
    if (ldo % 2 != 0) return fail(ZDT_EINVAL, "c2r: column stride must be even for even N");
    const FftPlan *pM = nullptr, *pN = nullptr;
    if (M > 1) {
      ZDT_TRY(fft_plan_get(M, false, &pM, maxr));
      if (fs_has(pM))  // the pre-pass on the first load
        return fs_run(pM, FS_C2R, in, ldi, out, ldo / 2, batch, true, scale / static_cast<double>(M),
                      static_cast<c32*>(s0), st);
    }
    ZDT_TRY(fft_plan_get(N, false, &pN, maxr));
    c32* Z = static_cast<c32*>(s2);
    {
      ProfScope ps(st, "c2r_pre", 16.0 * static_cast<double>(M * batch));
      c2r_pre<<<grid_for((M / 2 + 1) * batch, 256), 256, 0, st>>>(
          in, Z, static_cast<const c32*>(pN->tw), M, ldi, batch, static_cast<float>(scale / M));
      ZDT_CHECK_LAUNCH("c2r_pre");
    }
    if (M == 1) {
      ZDT_TRY_HIP(hipMemcpy2DAsync(out, ldo * sizeof(float), Z, sizeof(c32), sizeof(c32), batch,
                                   hipMemcpyDeviceToDevice, st));
    } else {
      ZDT_TRY(fft_plan_get(M, false, &pM, maxr));
      ZDT_TRY(fft_c2c(pM, Z, 1, M, out, 1, ldo / 2, batch, true, 1.0, s0, s1, st));
    }
    return ZDT_OK;
  }
  const FftPlan* p = nullptr;
  ZDT_TRY(fft_plan_get(N, false, &p, maxr));
  if (fs_has(p))
    return fs_run(p, FS_ODD_C2R, in, ldi, out, ldo, batch, true, scale / static_cast<double>(N),
                  static_cast<c32*>(s0), st, wide);
  c32* full = static_cast<c32*>(s2);
  hermitian_extend<<<grid_for(N * batch, 256), 256, 0, st>>>(in, ldi, full, N, batch);
  ZDT_CHECK_LAUNCH("hermitian_extend");
  ZDT_TRY(fft_c2c(p, full, 1, N, full, 1, N, batch, true, scale / static_cast<double>(N), s0, s1, st));
  complex_real_part<<<grid_for(N * batch, 256), 256, 0, st>>>(full, out, ldo, N, batch);
  ZDT_CHECK_LAUNCH("complex_real_part");
  return ZDT_OK;
}

__global__ void clear_wide(int64_t* wide) { *wide = 0; }

int fft_clear_wide(int64_t* wide, hipStream_t st) {
  clear_wide<<<1, 1, 0, st>>>(wide);
  ZDT_CHECK_LAUNCH("clear_wide");
  return ZDT_OK;
}

}  // namespace zdt
