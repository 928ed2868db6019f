// FFT convolution kernels for power-of-two frames with a precomputed PSF spectrum, hand-written for
// gfx950, templated on the complex type: float2 (fft.hip) and double2 (fft_f64.hip).
//
// Semantics follow the reference fft_convolve (pymoresane/iuwt_convolution.py:18-73):
//   linear   : out = crop_N(fftshift(irfft2(S * rfft2(pad_2N(x)))))
//   circular : out = fftshift(irfft2(S * rfft2(x)))
// Both are circular convolutions on a P x P frame (P = 2N or N) followed by a
// crop.  Here the image sits at the frame origin and the P/2 spatial roll
// that the shift/crop implies is folded into the PSF frame once, when the
// spectrum is built, so the output is simply the first N rows/columns.
//
// Passes (all FFTs run in LDS, radix-16/32 butterflies in registers):
//   1. rows r2c   : each image row (zero-padded to P) -> P/2+1 frequencies
//                   via a P/2-point complex FFT; written column-major
//                   (frequency k owns a contiguous column of rows).
//   2. columns    : per frequency column: forward P-point FFT (decimation in
//                   frequency, output left in digit-reversed order), pointwise
//                   product with the PSF column stored in that same order,
//                   inverse FFT (decimation in time, natural order out); only
//                   the N kept rows are written.  No reordering pass exists.
//   3. rows c2r   : per kept row: Hermitian pre-twiddle into a P/2-point
//                   inverse FFT, scale 1/P^2, write the N kept columns.
// Twiddles come from a device table exp(-2 pi i k / 2^14) computed on the
// host in double precision (float64 entries from 80-bit angles); float32
// in-butterfly powers are formed by a balanced product tree from one table
// value, float64 ones by at most one product of table values (see Twiddles).
#pragma once

#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>
#include <vector>

#include "pms_internal.h"

namespace pms {
namespace {

constexpr int kThreads = 256;

template <class C>
struct RealOf;
template <>
struct RealOf<float2> {
  using R = float;
};
template <>
struct RealOf<double2> {
  using R = double;
};
template <class C>
using Rl = typename RealOf<C>::R;

template <class C>
__device__ __forceinline__ C mk(Rl<C> x, Rl<C> y) {
  C r;
  r.x = x;
  r.y = y;
  return r;
}
template <class C>
__device__ __forceinline__ C cadd(C a, C b) {
  return mk<C>(a.x + b.x, a.y + b.y);
}
template <class C>
__device__ __forceinline__ C csub(C a, C b) {
  return mk<C>(a.x - b.x, a.y - b.y);
}
template <class C>
__device__ __forceinline__ C cmul(C a, C b) {
  return mk<C>(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}
template <class C>
__device__ __forceinline__ C cconj(C a) {
  return mk<C>(a.x, -a.y);
}
template <class C>
__device__ __forceinline__ C cscale(C a, Rl<C> s) {
  return mk<C>(a.x * s, a.y * s);
}

// the dynamic LDS as complex values
template <class C>
__device__ __forceinline__ C* dyn_lds() {
  extern __shared__ __align__(16) unsigned char fft_lds[];
  return reinterpret_cast<C*>(fft_lds);
}

// LDS index with one padding slot per 32 complex values (breaks power-of-two bank strides)
__device__ __forceinline__ int pad(int i) { return i + (i >> 5); }

// cos / sin of 2 pi j / 32 for j in [0, 16)
struct Roots32 {
  static constexpr double c[16] = {
      1.0, 0.9807852804032304, 0.9238795325112867, 0.8314696123025452,
      0.7071067811865476, 0.5555702330196022, 0.3826834323650898, 0.19509032201612828,
      0.0, -0.19509032201612828, -0.3826834323650898, -0.5555702330196022,
      -0.7071067811865476, -0.8314696123025452, -0.9238795325112867, -0.9807852804032304};
  static constexpr double s[16] = {
      0.0, 0.19509032201612828, 0.3826834323650898, 0.5555702330196022,
      0.7071067811865476, 0.8314696123025452, 0.9238795325112867, 0.9807852804032304,
      1.0, 0.9807852804032304, 0.9238795325112867, 0.8314696123025452,
      0.7071067811865476, 0.5555702330196022, 0.3826834323650898, 0.19509032201612828};
};

// t = o * exp(DIR * 2 pi i k / R), k < R/2 known at compile time after unrolling
template <class C, int R, int DIR>
__device__ __forceinline__ C rot(C o, int k) {
  const int j = k * (32 / R);
  if (j == 0) return o;
  if (j == 8) return DIR < 0 ? mk<C>(o.y, -o.x) : mk<C>(-o.y, o.x);
  const C w = mk<C>((Rl<C>)Roots32::c[j], (Rl<C>)(DIR * Roots32::s[j]));
  return cmul(o, w);
}

// In-register DFT: x_k <- sum_m x_m exp(DIR * 2 pi i m k / R), natural order in and out.
template <class C, int R, int DIR>
struct Dft {
  __device__ __forceinline__ static void run(C (&x)[R]) {
    C e[R / 2], o[R / 2];
#pragma unroll
    for (int k = 0; k < R / 2; ++k) {
      e[k] = x[2 * k];
      o[k] = x[2 * k + 1];
    }
    Dft<C, R / 2, DIR>::run(e);
    Dft<C, R / 2, DIR>::run(o);
#pragma unroll
    for (int k = 0; k < R / 2; ++k) {
      const C t = rot<C, R, DIR>(o[k], k);
      x[k] = cadd(e[k], t);
      x[k + R / 2] = csub(e[k], t);
    }
  }
};
template <class C, int DIR>
struct Dft<C, 1, DIR> {
  __device__ __forceinline__ static void run(C (&)[1]) {}
};

// The twiddles w^1 .. w^(R-1) of a butterfly, w = tw[i].  float32: all from w by a balanced product tree.
// float64: a power formed by squaring errs by its exponent's half in units of w's error, so w^1 .. w^3, w^4, w^8
// and w^12 come from the table and the others are one product of those.
template <class C, int R>
struct Twiddles {
  static constexpr bool kTree = sizeof(Rl<C>) == 4;
  static constexpr int N = kTree || R == 2 ? 1 : R == 4 ? 3 : R == 8 ? 4 : 6;
  static constexpr int exponent(int j) { return j < 4 ? j + 1 : 4 * (j - 2); }
  C w[N];
  __device__ __forceinline__ void load(const C* __restrict__ tw, int i) {
#pragma unroll
    for (int j = 0; j < N; ++j) w[j] = tw[exponent(j) * i];
  }
  __device__ __forceinline__ void none() {
#pragma unroll
    for (int j = 0; j < N; ++j) w[j] = mk<C>(1, 0);
  }
  template <bool CONJ>
  __device__ __forceinline__ void powers(C (&wk)[R]) const {
    const auto at = [&](int j) { return CONJ ? cconj(w[j]) : w[j]; };
    wk[0] = mk<C>(1, 0);
    wk[1] = at(0);
#pragma unroll
    for (int k = 2; k < R; ++k) {
      if (kTree)
        wk[k] = cmul(wk[k >> 1], wk[k - (k >> 1)]);
      else if (k < 4)
        wk[k] = at(k - 1);
      else if (k % 4 == 0)
        wk[k] = at(k / 4 + 2);
      else
        wk[k] = cmul(wk[k & ~3], wk[k & 3]);
    }
  }
};

// One in-place radix-R stage over an LDS array of length L, sub-transform
// length Ls (M = Ls/R).  Forward = decimation in frequency; inverse runs the
// exact mirror (conjugate twiddles before the butterfly).
template <class C, int R, bool FWD>
__device__ __forceinline__ void fft_stage(C* sm, int L, int Ls, int lt, int nthr, const C* tw) {
  const int M = Ls / R;
  const int mM = __ffs(M) - 1;  // M is a power of two
  const int nbf = L / R;
  const int tw_step = kFftMaxLen / Ls;
  for (int b = lt; b < nbf; b += nthr) {
    const int blk = b >> mM;
    const int n = b & (M - 1);
    const int base = blk * Ls + n;
    C x[R];
#pragma unroll
    for (int k = 0; k < R; ++k) x[k] = sm[pad(base + k * M)];
    if (FWD) {
      Dft<C, R, -1>::run(x);
      if (M > 1) {
        C wk[R];
        Twiddles<C, R> w;
        w.load(tw, n * tw_step);
        w.template powers<false>(wk);
#pragma unroll
        for (int k = 1; k < R; ++k) x[k] = cmul(x[k], wk[k]);
      }
    } else {
      if (M > 1) {
        C wk[R];
        Twiddles<C, R> w;
        w.load(tw, n * tw_step);
        w.template powers<true>(wk);
#pragma unroll
        for (int k = 1; k < R; ++k) x[k] = cmul(x[k], wk[k]);
      }
      Dft<C, R, +1>::run(x);
    }
#pragma unroll
    for (int k = 0; k < R; ++k) sm[pad(base + k * M)] = x[k];
  }
}

// Radix plan for L = 2^m: ns = ceil(m/4) stages, the first of radix 2^(m - 4(ns-1)) in {2,4,8,16},
// the rest radix 16.  Stage i (DIF order) works on sub-transforms of length Ls_i:
// Ls_0 = L, Ls_i = 16^(ns-i) for i >= 1.
__host__ __device__ __forceinline__ int plan_stages(int m) { return (m + 3) >> 2; }
__host__ __device__ __forceinline__ int plan_first_log2(int m) { return m - 4 * (plan_stages(m) - 1); }

// storage position of frequency k after the forward transform of length 2^m:
// k = d0 + R0 (d1 + 16 (d2 + ...)), position = d0 L/R0 + d1 L/(16 R0) + ...
__host__ __device__ __forceinline__ int perm_pos(int k, int m) {
  const int ns = plan_stages(m);
  const int lr0 = plan_first_log2(m);
  int mM = m - lr0;
  int pos = (k & ((1 << lr0) - 1)) << mM;
  k >>= lr0;
  for (int i = 1; i < ns; ++i) {
    mM -= 4;
    pos += (k & 15) << mM;
    k >>= 4;
  }
  return pos;
}

// ---- fused stage helpers --------------------------------------------------------------
// First DIF stage (radix R0, sub-transform length L, M0 = L/R0) fused with the load of the
// transform input: element e is fetched by get(e).  Batches of U butterflies are loaded before
// any is computed so that ~16 global loads per thread are in flight.
template <class C, int R0, class Get>
__device__ __forceinline__ void stage0_load(C* sm, int L, int lt, int nthr, const C* tw, Get get) {
  const int M0 = L / R0;
  const int step = kFftMaxLen / L;
  constexpr int U = (R0 >= 16) ? 1 : (R0 >= 8) ? 2 : (16 / R0);
  for (int n0 = lt; n0 < M0; n0 += nthr * U) {
    C x[U][R0];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = n0 + u * nthr;
#pragma unroll
      for (int k = 0; k < R0; ++k) x[u][k] = (n < M0) ? get(n + k * M0) : mk<C>(0, 0);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = n0 + u * nthr;
      if (n < M0) {
        Dft<C, R0, -1>::run(x[u]);
        if (M0 > 1) {
          C wk[R0];
          Twiddles<C, R0> w;
          w.load(tw, n * step);
          w.template powers<false>(wk);
#pragma unroll
          for (int k = 1; k < R0; ++k) x[u][k] = cmul(x[u][k], wk[k]);
        }
#pragma unroll
        for (int k = 0; k < R0; ++k) sm[pad(n + k * M0)] = x[u][k];
      }
    }
  }
}

// middle radix-16 stages i in [i0, i1) (forward) of an ns-stage plan: Ls = 16^(ns-i)
template <class C>
__device__ __forceinline__ void mid_forward(C* sm, int L, int ns, int i0, int i1, int lt, int nthr, const C* tw) {
  for (int i = i0; i < i1; ++i) {
    fft_stage<C, 16, true>(sm, L, 1 << (4 * (ns - i)), lt, nthr, tw);
    __syncthreads();
  }
}

// Per-job pointers of a batched launch (grid y selects the job), for NB = 1 or kMaxBatch jobs: see
// kMaxBatch on what the size of a launch's arguments costs.
template <class C, int NB>
struct R2cBatch {
  const void* src[NB];
  C* T[NB];
  const int* pred[NB];
};
template <class C, int NB>
struct ColBatch {
  const C* T1[NB];
  const C* S[NB];
  C* T2[NB];
  const int* pred[NB];
};
template <class C, int NB>
struct C2rBatch {
  const C* T2[NB];
  Rl<C>* out[NB];
  const int* pred[NB];
};

// ---- pass 1: rows r2c.  Group g of the block handles frame row fr; output T[k*ldT + fr], k in [0, P/2].
// The frame row is a row of the centred, rolled PSF (off = q/2).
template <class C, class TIN, int R0>
__global__ __launch_bounds__(kThreads) void k_rows_r2c(R2cBatch<C, 1> bt, int q, int off, int pm, int n_rows, int rb,
                                                       int ldT, const C* __restrict__ tw) {
  const int jb = blockIdx.y;
  const int* pred = bt.pred[jb];
  if (pred && *pred == 0) return;
  const TIN* __restrict__ src = static_cast<const TIN*>(bt.src[jb]);
  C* __restrict__ T = bt.T[jb];
  C* smem = dyn_lds<C>();
  const int P = 1 << pm;
  const int L = P >> 1;
  const int mL = pm - 1;
  const int nthr = kThreads / rb;
  const int g = threadIdx.x / nthr;
  const int lt = threadIdx.x - g * nthr;
  const int fr = xcd_remap(blockIdx.x, gridDim.x) * rb + g;
  C* sm = smem + g * (L + (L >> 5));
  const bool live = fr < n_rows;
  const int pmask = P - 1;
  const int a = (fr + off) & pmask;
  const bool row_ok = live && a < q;
  const TIN* row = src + (size_t)a * q;
  stage0_load<C, R0>(sm, L, lt, nthr, tw, [&](int e) {
    if (!row_ok) return mk<C>(0, 0);
    const int b0 = (2 * e + off) & pmask, b1 = (2 * e + 1 + off) & pmask;
    return mk<C>(b0 < q ? (Rl<C>)row[b0] : (Rl<C>)0, b1 < q ? (Rl<C>)row[b1] : (Rl<C>)0);
  });
  __syncthreads();
  mid_forward(sm, L, plan_stages(mL), 1, plan_stages(mL), lt, nthr, tw);
  if (!live) return;
  const int step = kFftMaxLen / P;
  for (int k = lt; k <= L; k += nthr) {
    const C zk = sm[pad(perm_pos(k & (L - 1), mL))];
    const C zl = cconj(sm[pad(perm_pos((L - k) & (L - 1), mL))]);
    const C e = cscale(cadd(zk, zl), 0.5f);
    const C dd = cscale(csub(zk, zl), 0.5f);
    const C o = mk<C>(dd.y, -dd.x);  // (zk - conj zl) / (2i)
    T[(size_t)k * ldT + fr] = cadd(e, cmul(tw[k * step], o));
  }
}

// ---- pass 2b: column forward FFT only (PSF spectrum), stored in the digit-reversed order
template <class C, int R0>
__global__ __launch_bounds__(kThreads) void k_cols_fwd(const C* __restrict__ T1, int pm, C* __restrict__ S, int cpb,
                                                       const C* __restrict__ tw) {
  C* smem = dyn_lds<C>();
  const int P = 1 << pm;
  const int ncols = (P >> 1) + 1;
  const int nthr = kThreads / cpb;
  const int g = threadIdx.x / nthr;
  const int lt = threadIdx.x - g * nthr;
  const int k = blockIdx.x * cpb + g;
  const bool live = k < ncols;
  C* sm = smem + g * (P + (P >> 5));
  const C* col = T1 + (size_t)k * P;
  stage0_load<C, R0>(sm, P, lt, nthr, tw, [&](int e) { return live ? col[e] : mk<C>(0, 0); });
  __syncthreads();
  mid_forward(sm, P, plan_stages(pm), 1, plan_stages(pm), lt, nthr, tw);
  if (!live) return;
  C* out = S + (size_t)k * P;
  for (int i = lt; i < P; i += nthr) out[i] = sm[pad(i)];
}

// =============================================================================================
// Convolution passes with compile-time plans.  For a frame of side P = 2^PG the radix plan, every
// LDS offset inside a butterfly and each thread's share of the work are constants, so the only
// per-butterfly integer work is one base address.  Every global operand a thread needs (stage-0
// inputs, in-stage twiddles, the PSF segment it multiplies with, the real-FFT post-processing
// twiddles) is requested at kernel start, so a kernel pays one memory latency instead of one per
// stage.  LIN marks the linear-convolution frame (P = 2N): half of every transform input is zero
// padding, and only half of every inverse output is kept.  Storage order, twiddles and arithmetic
// order per butterfly are those of the generic kernels above (same digit-reversed layout).

// LDS slot of element i: one pad per 32 and one more per 256 elements.  The second term spreads the
// digit-reversed (stride-256) accesses of the real-FFT split over all banks; both terms are linear
// over every butterfly's elements (base + k*M never carries into them), so a butterfly's offsets
// stay compile-time constants.  span() is a transform's LDS length, odd so that the transforms of
// one block start on different banks.
__host__ __device__ constexpr int padc(int i) { return i + (i >> 5) + (i >> 8); }
__host__ __device__ constexpr int span(int n) { return padc(n) + 1; }

template <int LG>
struct Plan {
  static constexpr int L = 1 << LG;
  static constexpr int NS = (LG + 3) >> 2;
  static constexpr int LR0 = LG - 4 * (NS - 1);
  static constexpr int R0 = 1 << LR0;
  static constexpr int M0 = L / R0;
  static constexpr int NBF = NS > 1 ? L / 16 : 0;  // radix-16 butterflies per stage
  static constexpr int ls(int i) { return 1 << (4 * (NS - i)); }
};

template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

template <int B, int E, class F>
__device__ __forceinline__ void static_for_down(F&& f) {  // E-1 down to B
  if constexpr (B < E) {
    f(std::integral_constant<int, E - 1>{});
    static_for_down<B, E - 1>(f);
  }
}

// This thread's in-stage twiddles for the radix-16 stages 1..NS-1 (butterflies b = lt + j*NT).
template <class C, int LG, int NT>
struct StageTw {
  using Pl = Plan<LG>;
  static constexpr int PER = Pl::NBF > 0 ? (Pl::NBF + NT - 1) / NT : 1;
  static constexpr int NI = Pl::NS > 1 ? Pl::NS : 1;
  Twiddles<C, 16> w[NI][PER];
  __device__ __forceinline__ void load(int lt, const C* __restrict__ gtw) {
    static_for<1, Pl::NS>([&](auto ic) {
      constexpr int I = decltype(ic)::value;
      constexpr int Ls = Pl::ls(I);
      constexpr int M = Ls / 16;
      if constexpr (M > 1) {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
          const int b = lt + j * NT;
          if (b < Pl::NBF)
            w[I][j].load(gtw, (b & (M - 1)) * (kFftMaxLen / Ls));
          else
            w[I][j].none();
        }
      }
    });
  }
};

// radix-16 stage I of one transform in LDS (sm), forward (DIF, twiddles after the butterfly) or
// inverse (the mirror: conjugate twiddles before the butterfly)
template <class C, int LG, int NT, int I, bool FWD>
__device__ __forceinline__ void stage16(C* sm, int lt, const StageTw<C, LG, NT>& tw) {
  using Pl = Plan<LG>;
  constexpr int Ls = Pl::ls(I);
  constexpr int M = Ls / 16;
  constexpr int LM = 4 * (Pl::NS - I - 1);
  constexpr int PER = StageTw<C, LG, NT>::PER;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int b = lt + j * NT;
    if ((Pl::NBF % NT) != 0 && b >= Pl::NBF) break;
    const int base = ((b >> LM) << (LM + 4)) + (b & (M - 1));
    C* s0 = sm + padc(base);
    C x[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) x[k] = s0[padc(k * M)];
    if constexpr (FWD) {
      Dft<C, 16, -1>::run(x);
      if constexpr (M > 1) {
        C wk[16];
        tw.w[I][j].template powers<false>(wk);
#pragma unroll
        for (int k = 1; k < 16; ++k) x[k] = cmul(x[k], wk[k]);
      }
    } else {
      if constexpr (M > 1) {
        C wk[16];
        tw.w[I][j].template powers<true>(wk);
#pragma unroll
        for (int k = 1; k < 16; ++k) x[k] = cmul(x[k], wk[k]);
      }
      Dft<C, 16, +1>::run(x);
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) s0[padc(k * M)] = x[k];
  }
}

// stage 0 (radix R0) inputs of this thread: butterflies n = lt + u*NT < M0, elements n + k*M0;
// KL of the R0 inputs are non-zero (LIN: the upper half is zero padding)
template <class C, int LG, int NT, bool LIN>
struct Stage0 {
  using Pl = Plan<LG>;
  static constexpr int U = (Pl::M0 + NT - 1) / NT;
  static constexpr int KL = LIN ? (Pl::R0 / 2 > 0 ? Pl::R0 / 2 : 1) : Pl::R0;
  C x[U][Pl::R0];
  Twiddles<C, Pl::R0> w[U];
  template <class Get>
  __device__ __forceinline__ void load(int lt, const C* __restrict__ gtw, Get get) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = lt + u * NT;
      const bool ok = n < Pl::M0;
#pragma unroll
      for (int k = 0; k < Pl::R0; ++k) x[u][k] = (ok && k < KL) ? get(n + k * Pl::M0) : mk<C>(0, 0);
      if constexpr (Pl::M0 > 1) {
        if (ok)
          w[u].load(gtw, n * (kFftMaxLen / Pl::L));
        else
          w[u].none();
      }
    }
  }
  // forward stage 0 from registers into LDS
  __device__ __forceinline__ void forward(C* sm, int lt) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = lt + u * NT;
      if ((Pl::M0 % NT) != 0 && n >= Pl::M0) break;
      Dft<C, Pl::R0, -1>::run(x[u]);
      if constexpr (Pl::M0 > 1) {
        C wk[Pl::R0];
        w[u].template powers<false>(wk);
#pragma unroll
        for (int k = 1; k < Pl::R0; ++k) x[u][k] = cmul(x[u][k], wk[k]);
      }
      C* s0 = sm + padc(n);
#pragma unroll
      for (int k = 0; k < Pl::R0; ++k) s0[padc(k * Pl::M0)] = x[u][k];
    }
  }
  // inverse last stage from LDS to put(e, value), keeping the first KL outputs of each butterfly
  template <class Put>
  __device__ __forceinline__ void inverse(const C* sm, int lt, Put put) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = lt + u * NT;
      if ((Pl::M0 % NT) != 0 && n >= Pl::M0) break;
      const C* s0 = sm + padc(n);
      C y[Pl::R0];
#pragma unroll
      for (int k = 0; k < Pl::R0; ++k) y[k] = s0[padc(k * Pl::M0)];
      if constexpr (Pl::M0 > 1) {
        C wk[Pl::R0];
        w[u].template powers<true>(wk);
#pragma unroll
        for (int k = 1; k < Pl::R0; ++k) y[k] = cmul(y[k], wk[k]);
      }
      Dft<C, Pl::R0, +1>::run(y);
#pragma unroll
      for (int k = 0; k < KL; ++k) put(n + k * Pl::M0, y[k]);
    }
  }
};

// points per thread in the row and column transforms: 32 in float32 (measured at P = 8192: 32 points per
// thread beats 16, whose extra threads buy occupancy but not speed), 16 in float64, the same registers
#ifndef PMS_FFT_PTS
#define PMS_FFT_PTS 32
#endif
template <class C>
constexpr int kFftPts = PMS_FFT_PTS * 4 / (int)sizeof(Rl<C>);

// launch shapes, functions of the frame only
// Rows: NT threads per row (at most kFftPts points each, at least one wave), RB rows per block as many as
// 512 threads, ~140 KB of LDS and >= 256 blocks allow: more rows per block make longer contiguous
// runs in the transposed (column-major) writes and reads.
template <class C, int PG, bool LIN>
struct RowCfg {
  static constexpr int P = 1 << PG, L = P / 2, N = LIN ? L : P;  // N = rows = image side
  static constexpr int NT = (L / kFftPts<C> > 64) ? L / kFftPts<C> : 64;
  static constexpr int rb() {
    int r = 16;
    while (r > 1 && (r * NT > 512 || (size_t)r * span(L) * sizeof(C) > 140 * 1024 || N / r < 256))
      r >>= 1;
    return r;
  }
  static constexpr int RB = rb();
  static constexpr int T = RB * NT;
  static constexpr int NPP = (RB * (L / 2 + 1) + T - 1) / T;  // real-FFT pairs per thread
  static constexpr size_t LDS = (size_t)RB * span(L) * sizeof(C);
};

template <class C, int PG>
struct ColCfg {
  static constexpr int P = 1 << PG;
  static constexpr int cpb() {
    int c = 256 * kFftPts<C> / P;
    if (c > 16) c = 16;
    if (c < 1) c = 1;
    while (c > 1 && (P / 2 + 1) / c < 256) c >>= 1;
    return c;
  }
  static constexpr int CPB = cpb();
  static constexpr int NT = (P / (256 / CPB) > kFftPts<C>) ? P / kFftPts<C> : 256 / CPB;
  static constexpr int T = CPB * NT;
  static constexpr size_t LDS = (size_t)CPB * span(P) * sizeof(C);
};

// storage position of frequency k (compile-time plan of length 2^LG)
template <int LG>
__device__ __forceinline__ int pos_of(int k) {
  using Pl = Plan<LG>;
  int mM = LG - Pl::LR0;
  int pos = (k & (Pl::R0 - 1)) << mM;
  k >>= Pl::LR0;
#pragma unroll
  for (int i = 1; i < Pl::NS; ++i) {
    mM -= 4;
    pos += (k & 15) << mM;
    k >>= 4;
  }
  return pos;
}

// ---- pass 1: rows r2c.  Block = RB frame rows; output T[k*ldT + row], k in [0, P/2].
template <class C, int PG, bool LIN, int NB>
__global__ __launch_bounds__((RowCfg<C, PG, LIN>::T)) void k_conv_r2c(R2cBatch<C, NB> bt, int n_rows, int ldT,
                                                                      const C* __restrict__ tw) {
  using G = RowCfg<C, PG, LIN>;
  constexpr int LG = PG - 1;
  constexpr int L = G::L, RB = G::RB, NT = G::NT, SP = span(L);
  const int jb = blockIdx.y;
  const int* pred = bt.pred[jb];
  if (pred && *pred == 0) return;
  const Rl<C>* __restrict__ src = static_cast<const Rl<C>*>(bt.src[jb]);
  C* __restrict__ T = bt.T[jb];
  C* smem = dyn_lds<C>();
  const int g = threadIdx.x / NT;
  const int lt = threadIdx.x - g * NT;
  const int row0 = xcd_remap(blockIdx.x, gridDim.x) * RB;
  const int fr = row0 + g;
  const bool live = fr < n_rows;
  C* sm = smem + g * SP;
  // everything global this thread needs, requested up front
  const Rl<C>* row = src + (size_t)(live ? fr : 0) * G::N;
  Stage0<C, LG, NT, LIN> s0;
  s0.load(lt, tw, [&](int e) { return live ? *reinterpret_cast<const C*>(row + 2 * e) : mk<C>(0, 0); });
  StageTw<C, LG, NT> stw;
  stw.load(lt, tw);
  constexpr int step = kFftMaxLen / (2 * L);
  C wpp[G::NPP];
#pragma unroll
  for (int i = 0; i < G::NPP; ++i) {
    const int idx = threadIdx.x + i * G::T;
    const int k = idx / RB;
    wpp[i] = (k <= L / 2) ? tw[k * step] : mk<C>(1, 0);
  }
  s0.forward(sm, lt);
  __syncthreads();
  static_for<1, Plan<LG>::NS>([&](auto ic) {
    stage16<C, LG, NT, decltype(ic)::value, true>(sm, lt, stw);
    __syncthreads();
  });
  // Hermitian split of the packed transform: X[k], X[L-k] from Z[k], Z[L-k]; consecutive threads
  // take consecutive rows of one k so the transposed writes pair up
#pragma unroll
  for (int i = 0; i < G::NPP; ++i) {
    const int idx = threadIdx.x + i * G::T;
    const int k = idx / RB;
    const int g2 = idx - k * RB;
    const int r2 = row0 + g2;
    if (k > L / 2 || r2 >= n_rows) continue;
    const C* sm2 = smem + g2 * SP;
    const int pk = pos_of<LG>(k & (L - 1)), pl = pos_of<LG>((L - k) & (L - 1));
    const C zk = sm2[padc(pk)];
    const C zl = sm2[padc(pl)];
    const C w = wpp[i];
    {
      const C c = cconj(zl);
      const C e = cscale(cadd(zk, c), (Rl<C>)0.5);
      const C dd = cscale(csub(zk, c), (Rl<C>)0.5);
      T[(size_t)k * ldT + r2] = cadd(e, cmul(w, mk<C>(dd.y, -dd.x)));
    }
    if (k != L - k) {
      const C c = cconj(zk);
      const C e = cscale(cadd(zl, c), (Rl<C>)0.5);
      const C dd = cscale(csub(zl, c), (Rl<C>)0.5);
      const C wl = mk<C>(-w.x, w.y);  // w^(L-k) = -conj(w^k)
      T[(size_t)(L - k) * ldT + r2] = cadd(e, cmul(wl, mk<C>(dd.y, -dd.x)));
    }
  }
}

// ---- pass 2: column convolution: forward FFT, product with the PSF column, inverse FFT.
template <class C, int PG, bool LIN, int NB>
__global__ __launch_bounds__((ColCfg<C, PG>::T)) void k_conv_cols(ColBatch<C, NB> bt, int n_rows,
                                                               const C* __restrict__ tw) {
  using G = ColCfg<C, PG>;
  using Pl = Plan<PG>;
  constexpr int P = G::P, NT = G::NT, SP = span(P);
  constexpr int NCOLS = P / 2 + 1;
  const int jb = blockIdx.y;
  const int* pred = bt.pred[jb];
  if (pred && *pred == 0) return;
  C* smem = dyn_lds<C>();
  const int g = threadIdx.x / NT;
  const int lt = threadIdx.x - g * NT;
  const int k = blockIdx.x * G::CPB + g;
  const bool live = k < NCOLS;
  C* sm = smem + g * SP;
  const C* __restrict__ col = bt.T1[jb] + (size_t)(live ? k : 0) * n_rows;
  const C* __restrict__ sc = bt.S[jb] + (size_t)(live ? k : 0) * P;
  C* __restrict__ out = bt.T2[jb] + (size_t)(live ? k : 0) * n_rows;
  if constexpr (Pl::NS == 1) {
    // whole transform in one thread's registers (P <= 16)
    if (!live || lt != 0) return;
    C x[P];
#pragma unroll
    for (int e = 0; e < P; ++e) x[e] = (!LIN || e < P / 2) ? col[e] : mk<C>(0, 0);
    Dft<C, P, -1>::run(x);
#pragma unroll
    for (int e = 0; e < P; ++e) x[e] = cmul(x[e], sc[e]);
    Dft<C, P, +1>::run(x);
#pragma unroll
    for (int e = 0; e < (LIN ? P / 2 : P); ++e) out[e] = x[e];
  } else {
    Stage0<C, PG, NT, LIN> s0;
    // unconditional loads (a dead block reads column 0 and stores nothing): loads under a branch
    // leave the compiler's wait counts conservative, so that stage 0 would also wait for the PSF
    // segment requested after its inputs
    s0.load(lt, tw, [&](int e) { return col[e]; });
    StageTw<C, PG, NT> stw;
    stw.load(lt, tw);
    constexpr int PER = StageTw<C, PG, NT>::PER;
    C sv[PER][16];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int b = lt + j * NT;
#pragma unroll
      for (int m = 0; m < 16; ++m) sv[j][m] = (b < Pl::NBF) ? sc[16 * b + m] : mk<C>(0, 0);
    }
    s0.forward(sm, lt);
    __syncthreads();
    static_for<1, Pl::NS - 1>([&](auto ic) {
      stage16<C, PG, NT, decltype(ic)::value, true>(sm, lt, stw);
      __syncthreads();
    });
    // last forward stage (sub-length 16), PSF product, first inverse stage, in registers
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int b = lt + j * NT;
      if ((Pl::NBF % NT) != 0 && b >= Pl::NBF) break;
      const int base = 16 * b;
      C* s1 = sm + padc(base);
      C x[16];
#pragma unroll
      for (int m = 0; m < 16; ++m) x[m] = s1[m];
      Dft<C, 16, -1>::run(x);
#pragma unroll
      for (int m = 0; m < 16; ++m) x[m] = cmul(x[m], sv[j][m]);
      Dft<C, 16, +1>::run(x);
#pragma unroll
      for (int m = 0; m < 16; ++m) s1[m] = x[m];
    }
    __syncthreads();
    static_for_down<1, Pl::NS - 1>([&](auto ic) {
      stage16<C, PG, NT, decltype(ic)::value, false>(sm, lt, stw);
      __syncthreads();
    });
    if (!live) return;
    s0.inverse(sm, lt, [&](int e, C v) { out[e] = v; });
  }
}

// ---- pass 3: rows c2r.  Block = RB kept rows; out[r * N + c].
template <class C, int PG, bool LIN, int NB>
__global__ __launch_bounds__((RowCfg<C, PG, LIN>::T)) void k_conv_c2r(C2rBatch<C, NB> bt, int n_rows, int ldT, Rl<C> scale,
                                                                      const C* __restrict__ tw) {
  using G = RowCfg<C, PG, LIN>;
  constexpr int LG = PG - 1;
  constexpr int L = G::L, RB = G::RB, NT = G::NT, SP = span(L);
  const int jb = blockIdx.y;
  const int* pred = bt.pred[jb];
  if (pred && *pred == 0) return;
  const C* __restrict__ T2 = bt.T2[jb];
  Rl<C>* __restrict__ out = bt.out[jb];
  C* smem = dyn_lds<C>();
  const int g = threadIdx.x / NT;
  const int lt = threadIdx.x - g * NT;
  const int row0 = xcd_remap(blockIdx.x, gridDim.x) * RB;
  const int r = row0 + g;
  const bool live = r < n_rows;
  C* sm = smem + g * SP;
  constexpr int step = kFftMaxLen / (2 * L);
  C xk[G::NPP], xl[G::NPP], wpp[G::NPP];
#pragma unroll
  for (int i = 0; i < G::NPP; ++i) {
    const int idx = threadIdx.x + i * G::T;
    const int k = idx / RB;
    const int r2 = row0 + (idx - k * RB);
    const bool ok = k <= L / 2 && r2 < n_rows;
    xk[i] = ok ? T2[(size_t)k * ldT + r2] : mk<C>(0, 0);
    xl[i] = ok ? T2[(size_t)(L - k) * ldT + r2] : mk<C>(0, 0);
    wpp[i] = ok ? tw[k * step] : mk<C>(1, 0);
  }
  StageTw<C, LG, NT> stw;
  stw.load(lt, tw);
  Stage0<C, LG, NT, LIN> s0;
  if constexpr (Plan<LG>::M0 > 1) {
#pragma unroll
    for (int u = 0; u < Stage0<C, LG, NT, LIN>::U; ++u) {
      const int n = lt + u * NT;
      if (n < Plan<LG>::M0)
        s0.w[u].load(tw, n * (kFftMaxLen / L));
      else
        s0.w[u].none();
    }
  }
  // Hermitian pre-twiddle: Z'[k] = (X[k] + conj X[L-k]) + i (X[k] - conj X[L-k]) conj(w^k), stored
  // digit-reversed for the inverse transform
#pragma unroll
  for (int i = 0; i < G::NPP; ++i) {
    const int idx = threadIdx.x + i * G::T;
    const int k = idx / RB;
    const int g2 = idx - k * RB;
    if (k > L / 2 || row0 + g2 >= n_rows) continue;
    C* sm2 = smem + g2 * SP;
    const C w = wpp[i];
    {
      const C e = cadd(xk[i], cconj(xl[i]));
      const C o = cmul(csub(xk[i], cconj(xl[i])), cconj(w));
      const int pk = pos_of<LG>(k & (L - 1));
      sm2[padc(pk)] = mk<C>(e.x - o.y, e.y + o.x);
    }
    const int kl = L - k;
    if (kl != k && kl < L) {
      const C e = cadd(xl[i], cconj(xk[i]));
      const C o = cmul(csub(xl[i], cconj(xk[i])), mk<C>(-w.x, -w.y));  // conj(w^(L-k)) = -w^k
      const int pl = pos_of<LG>(kl);
      sm2[padc(pl)] = mk<C>(e.x - o.y, e.y + o.x);
    }
  }
  __syncthreads();
  static_for_down<1, Plan<LG>::NS>([&](auto ic) {
    stage16<C, LG, NT, decltype(ic)::value, false>(sm, lt, stw);
    __syncthreads();
  });
  if (!live) return;
  Rl<C>* orow = out + (size_t)r * G::N;
  s0.inverse(sm, lt, [&](int e, C v) {
    *reinterpret_cast<C*>(orow + 2 * e) = mk<C>(v.x * scale, v.y * scale);
  });
}

template <class C, int PG, bool LIN, int NB>
void set_conv_attrs_nb(int lds_max) {
  (void)hipFuncSetAttribute((const void*)k_conv_r2c<C, PG, LIN, NB>, hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
  (void)hipFuncSetAttribute((const void*)k_conv_cols<C, PG, LIN, NB>, hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
  (void)hipFuncSetAttribute((const void*)k_conv_c2r<C, PG, LIN, NB>, hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
}

template <class C, int PG, bool LIN>
void set_conv_attrs(int lds_max) {
  set_conv_attrs_nb<C, PG, LIN, 1>(lds_max);
  set_conv_attrs_nb<C, PG, LIN, kMaxBatch>(lds_max);
}

template <class C, int PG, bool LIN, int NB>
void launch_conv(const R2cBatch<C, NB>& rb, const ColBatch<C, NB>& cb, const C2rBatch<C, NB>& ob, int nb, int n,
                 Rl<C> scale, const C* tw, hipStream_t st) {
  using R = RowCfg<C, PG, LIN>;
  using G = ColCfg<C, PG>;
  hipLaunchKernelGGL((k_conv_r2c<C, PG, LIN, NB>), dim3((n + R::RB - 1) / R::RB, nb), dim3(R::T), R::LDS, st, rb, n, n, tw);
  PMS_LAUNCH_CHECK();
  hipLaunchKernelGGL((k_conv_cols<C, PG, LIN, NB>), dim3((G::P / 2 + 1 + G::CPB - 1) / G::CPB, nb), dim3(G::T), G::LDS, st,
                     cb, n, tw);
  PMS_LAUNCH_CHECK();
  hipLaunchKernelGGL((k_conv_c2r<C, PG, LIN, NB>), dim3((n + R::RB - 1) / R::RB, nb), dim3(R::T), R::LDS, st, ob, n, n,
                     scale, tw);
  PMS_LAUNCH_CHECK();
}

template <class C, bool LIN, int NB>
void dispatch_conv(int pg, const R2cBatch<C, NB>& rb, const ColBatch<C, NB>& cb, const C2rBatch<C, NB>& ob, int nb,
                   int n, Rl<C> scale, const C* tw, hipStream_t st) {
  switch (pg) {
    case 2: launch_conv<C, 2, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st); break;
    case 3: launch_conv<C, 3, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st); break;
    case 4: launch_conv<C, 4, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st); break;
    case 5: launch_conv<C, 5, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st); break;
    case 6: launch_conv<C, 6, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st); break;
    case 7: launch_conv<C, 7, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st); break;
    case 8: launch_conv<C, 8, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st); break;
    case 9: launch_conv<C, 9, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st); break;
    case 10: launch_conv<C, 10, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st); break;
    case 11: launch_conv<C, 11, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st); break;
    case 12: launch_conv<C, 12, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st); break;
    case 13: launch_conv<C, 13, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st); break;
    case 14:
      if constexpr (sizeof(Rl<C>) == 4) {  // one LDS transform holds a column: 8192 in float64
        launch_conv<C, 14, LIN, NB>(rb, cb, ob, nb, n, scale, tw, st);
        break;
      }
      [[fallthrough]];
    default: fail(PMS_ERR_ARG, "FFT frame out of range");
  }
}

template <class C, bool LIN>
void set_all_conv_attrs(int lds_max) {
  set_conv_attrs<C, 2, LIN>(lds_max);
  set_conv_attrs<C, 3, LIN>(lds_max);
  set_conv_attrs<C, 4, LIN>(lds_max);
  set_conv_attrs<C, 5, LIN>(lds_max);
  set_conv_attrs<C, 6, LIN>(lds_max);
  set_conv_attrs<C, 7, LIN>(lds_max);
  set_conv_attrs<C, 8, LIN>(lds_max);
  set_conv_attrs<C, 9, LIN>(lds_max);
  set_conv_attrs<C, 10, LIN>(lds_max);
  set_conv_attrs<C, 11, LIN>(lds_max);
  set_conv_attrs<C, 12, LIN>(lds_max);
  set_conv_attrs<C, 13, LIN>(lds_max);
  if constexpr (sizeof(Rl<C>) == 4) set_conv_attrs<C, 14, LIN>(lds_max);
}

int env_int(const char* name, int dflt) {
  const char* v = getenv(name);
  return v ? atoi(v) : dflt;
}

// Rows / columns per workgroup of the PSF transform: as many as the LDS budget allows for wide coalesced
// row accesses, but never so many that the launch has fewer than ~256 workgroups (small frames stay
// parallel).  The budget counts float32 values; float64 ones take twice their LDS.
template <class C>
int rows_per_block(int L, int n_rows) {
  static const int lim = env_int("PMS_FFT_ROW_LDS", 8192) * (int)sizeof(float2) / (int)sizeof(C);
  int rb = lim / (L > 0 ? L : 1);
  if (rb > 16) rb = 16;
  while (rb > 1 && n_rows / rb < 256) rb >>= 1;
  if (rb < 1) rb = 1;
  return rb;
}

template <class C>
int cols_per_block(int P) {
  const int ncols = P / 2 + 1;
  int c = 8192 * (int)sizeof(float2) / (int)sizeof(C) / P;
  if (c > 16) c = 16;
  while (c > 1 && ncols / c < 256) c >>= 1;
  if (c < 1) c = 1;
  return c;
}

// first-stage radix of the plan for length 2^m
int first_radix(int m) { return 1 << plan_first_log2(m); }

// calls f(integral constant of the first-stage radix)
template <class F>
void with_radix(int r, F f) {
  switch (r) {
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    default: f(std::integral_constant<int, 16>{}); break;
  }
}

// The twiddle table exp(-2 pi i k / kFftMaxLen) of a device in complex type C, computed in float64; its first
// request also allows the kernels the large dynamic LDS (67.6 KB at P = 8192 in float32) that CDNA4's 160 KB permits.
template <class C>
struct Pow2Tables {
  std::mutex mu;
  C* ptr[64] = {};

  const C* get(int device) {
    PMS_REQUIRE(device >= 0 && device < 64, "device id out of range");
    std::lock_guard<std::mutex> lk(mu);
    if (ptr[device]) return ptr[device];
    std::vector<C> h(kFftMaxLen);
    for (int k = 0; k < kFftMaxLen; ++k) {
      // float64 entries from a wider angle, whose rounding would otherwise reach them
      using A = std::conditional_t<sizeof(Rl<C>) == 8, long double, double>;
      const A a = -2 * (A)M_PIl * (A)k / (A)kFftMaxLen;
      h[k].x = (Rl<C>)std::cos(a);
      h[k].y = (Rl<C>)std::sin(a);
    }
    const int lds_max = 160 * 1024;
    for (int r : {2, 4, 8, 16})
      with_radix(r, [&](auto rc) {
        constexpr int R0 = decltype(rc)::value;
        (void)hipFuncSetAttribute((const void*)k_rows_r2c<C, float, R0>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  lds_max);
        if constexpr (sizeof(Rl<C>) == 8)
          (void)hipFuncSetAttribute((const void*)k_rows_r2c<C, double, R0>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    lds_max);
        (void)hipFuncSetAttribute((const void*)k_cols_fwd<C, R0>, hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
      });
    set_all_conv_attrs<C, true>(lds_max);
    set_all_conv_attrs<C, false>(lds_max);
    (void)hipGetLastError();
    C* d = nullptr;
    PMS_HIP(hipMalloc(&d, sizeof(C) * kFftMaxLen));
    PMS_HIP(hipMemcpy(d, h.data(), sizeof(C) * kFftMaxLen, hipMemcpyHostToDevice));
    ptr[device] = d;
    return d;
  }
  const C* get() {
    int dev = 0;
    PMS_HIP(hipGetDevice(&dev));
    return get(dev);
  }
};

// spectrum of a q x q PSF centred in a p x p frame; work holds the (P/2+1) x P row spectra, column-major
template <class C, class TIN>
void pow2_psf_spectrum(const TIN* psf, int q, int p, C* spec, C* work, const C* tw, hipStream_t st) {
  const int pm = ilog2(p);
  const int L = p / 2;
  R2cBatch<C, 1> rb{};
  rb.src[0] = psf;
  rb.T[0] = work;
  const int rpb = rows_per_block<C>(L, p);
  const size_t lds1 = (size_t)rpb * (L + (L >> 5)) * sizeof(C);
  with_radix(first_radix(pm - 1), [&](auto rc) {
    hipLaunchKernelGGL((k_rows_r2c<C, TIN, decltype(rc)::value>), dim3(ceil_div(p, rpb), 1), dim3(kThreads), lds1, st,
                       rb, q, q / 2, pm, p, rpb, p, tw);
  });
  PMS_LAUNCH_CHECK();
  const int cpb = cols_per_block<C>(p);
  const size_t lds2 = (size_t)cpb * (p + (p >> 5)) * sizeof(C);
  with_radix(first_radix(pm), [&](auto rc) {
    hipLaunchKernelGGL((k_cols_fwd<C, decltype(rc)::value>), dim3(ceil_div(L + 1, cpb)), dim3(kThreads), lds2, st,
                       (const C*)work, pm, spec, cpb, tw);
  });
  PMS_LAUNCH_CHECK();
}

// nb <= NB jobs in one launch per pass.  Jobs are independent: job j's blocks read and write only job j's
// buffers, so a batch gives each job exactly the result of its own single-job call.
template <class C, int NB, class JOB>
void pow2_conv_jobs(const JOB* jobs, int nb, int n, int p, const C* tw, hipStream_t st) {
  const int pm = ilog2(p);
  const int L = p / 2;
  const Rl<C> scale = (Rl<C>)1 / ((Rl<C>)p * (Rl<C>)p);
  R2cBatch<C, NB> rb{};
  ColBatch<C, NB> cb{};
  C2rBatch<C, NB> ob{};
  for (int k = 0; k < nb; ++k) {
    const JOB& j = jobs[k];
    PMS_REQUIRE(j.in && j.spec && j.out && j.work, "fft_conv: NULL buffer");
    C* T1 = reinterpret_cast<C*>(j.work);
    C* T2 = T1 + (size_t)(L + 1) * n;
    rb.src[k] = j.in;
    rb.T[k] = T1;
    rb.pred[k] = j.pred;
    cb.T1[k] = T1;
    cb.S[k] = reinterpret_cast<const C*>(j.spec);
    cb.T2[k] = T2;
    cb.pred[k] = j.pred;
    ob.T2[k] = T2;
    ob.out[k] = j.out;
    ob.pred[k] = j.pred;
  }
  if (p == 2 * n)
    dispatch_conv<C, true, NB>(pm, rb, cb, ob, nb, n, scale, tw, st);
  else
    dispatch_conv<C, false, NB>(pm, rb, cb, ob, nb, n, scale, tw, st);
}

template <class C, class JOB>
void pow2_conv_batch(const JOB* jobs, int count, int n, int p, const C* tw, hipStream_t st) {
  PMS_REQUIRE(p == n || p == 2 * n, "fft_conv: frame must be N (circular) or 2N (linear)");
  for (int j0 = 0; j0 < count; j0 += kMaxBatch) {
    const int nb = std::min(kMaxBatch, count - j0);
    if (nb == 1)
      pow2_conv_jobs<C, 1>(jobs + j0, nb, n, p, tw, st);
    else
      pow2_conv_jobs<C, kMaxBatch>(jobs + j0, nb, n, p, tw, st);
  }
}

}  // namespace
}  // namespace pms
