// FFT convolution for any even frame side and for float64, hand-written for gfx950.
//
// Same three-pass structure and the same semantics as the power-of-two float32 kernels
// (fft.hip, reference pymoresane/iuwt_convolution.py:18-73): rows r2c -> column pass (forward,
// PSF product, inverse) -> rows c2r with scale and crop, the image at the frame origin and the
// P/2 roll folded into the PSF frame.  Differences: the transforms are mixed radix (prime
// factors up to 13) with the radix plan chosen at run time, and every kernel is templated on the
// arithmetic type, so this file serves frames whose side is not a power of two (the reference's
// numpy rfft2 takes any size, iuwt_convolution.py:64-73) in float32 and in float64 (the
// deconvolution's float64 precision mode).
//
// Each transform of length L runs in LDS as in-place decimation-in-frequency stages (forward,
// output in mixed-radix digit-reversed order) or their exact mirror (inverse, decimation in time,
// digit-reversed in, natural order out), so the column pass needs no reordering: the PSF
// spectrum is stored in the order in which the column pass multiplies by it.  The stages (radix 2 to 13)
// follow from the length; the host groups them into steps of one or two, which are compiled.  Stage twiddles, split factors
// and the row transforms' digit reversal come from tables per frame side and type, computed on the host in float64.
//
// What bounds the passes is the chain of each block: its loads, one LDS exchange and barrier per step, its
// stores.  So two stages that fit the registers are one step, the first and last steps work on global memory,
// twiddles and the PSF column are requested ahead of the barriers, nothing divides by a run-time number, and
// the blocks are small enough for 16 waves a CU.  Steps of 15 and 16 elements save more exchanges than they are
// worth (registers: 47 against 43 us in the mean below), and so does every other arithmetic: single-precision cleans
// amplify a rounding, so sums and products stay those of the separate stages (composite DFTs of 6 to
// 16 points were 37 us, no less exact, but moved a 120^2 clean by 3e-4).  Convolution of a 1000^2 image on a frame
// of 2000: 88 us with a division per butterfly, run-time digit reversal, an exchange per stage and two rows a
// block, 38 us now; frames of 132 / 800 / 3000 / 6000: 39 / 50 / 180 / 719 -> 21 / 23 / 75 / 256 us; geometric mean over 23 frames
// 96 -> 43 us.
#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <type_traits>
#include <vector>

#include "pms_internal.h"

namespace pms {
namespace {

constexpr int kGThreads = 512;

template <class T>
__device__ __forceinline__ Cx<T> cmk(T a, T b) {
  Cx<T> r;
  r.x = a;
  r.y = b;
  return r;
}
template <class T>
__device__ __forceinline__ Cx<T> gadd(Cx<T> a, Cx<T> b) {
  return cmk<T>(a.x + b.x, a.y + b.y);
}
template <class T>
__device__ __forceinline__ Cx<T> gsub(Cx<T> a, Cx<T> b) {
  return cmk<T>(a.x - b.x, a.y - b.y);
}
template <class T>
__device__ __forceinline__ Cx<T> gmul(Cx<T> a, Cx<T> b) {
  return cmk<T>(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}
template <class T>
__device__ __forceinline__ Cx<T> gconj(Cx<T> a) {
  return cmk<T>(a.x, -a.y);
}
template <class T>
__device__ __forceinline__ Cx<T> gscale(Cx<T> a, T s) {
  return cmk<T>(a.x * s, a.y * s);
}
// multiply by -i (forward) or +i (inverse)
template <class T, bool FWD>
__device__ __forceinline__ Cx<T> gmul_i(Cx<T> a) {
  return FWD ? cmk<T>(a.y, -a.x) : cmk<T>(-a.y, a.x);
}

// LDS slot of element i (one padding slot per 32 elements)
__device__ __forceinline__ int gpad(int i) { return i + (i >> 5); }
__host__ __device__ __forceinline__ int gspan(int n) { return n + (n >> 5) + 1; }

constexpr int kMaxSteps = 8;

// A step of a transform: one decimation-in-frequency stage of radix r1, or (r2 > 1) two successive stages in
// registers, r1 then r2, on the same r1 * r2 elements.
struct GStep {
  int r1, r2;
};
constexpr int kStepKinds = 12;
__host__ __device__ constexpr GStep step_kind(int k) {
  constexpr GStep t[kStepKinds] = {{2, 1}, {3, 1}, {4, 1}, {5, 1}, {7, 1}, {8, 1}, {11, 1}, {13, 1},
                                   {2, 3}, {2, 5}, {3, 3}, {4, 3}};
  return t[k];
}

// Plan of one transform length: step i works on sub-transforms of length Ls_i = L / (r(0) ... r(i-1)), r(i)
// the product of its radices.  Four bits a step: kernel arguments stay small.
struct GPlan {
  int L;
  int ns;
  uint32_t code;
  __host__ __device__ __forceinline__ int kind(int i) const { return (int)((code >> (4 * i)) & 15u); }
  __host__ __device__ __forceinline__ int r(int i) const { return step_kind(kind(i)).r1 * step_kind(kind(i)).r2; }
};

// Position of frequency k in the digit-reversed output of the forward transform, over its stages:
// k = d0 + r0 (d1 + r1 (d2 + ...)), position = d0 L/r0 + d1 L/(r0 r1) + ...
int gperm(const GPlan& p, int k) {
  int pos = 0, span = p.L;
  for (int i = 0; i < p.ns; ++i) {
    const GStep st = step_kind(p.kind(i));
    for (int r : {st.r1, st.r2}) {
      span /= r;
      const int q = k / r;
      pos += (k - q * r) * span;
      k = q;
    }
  }
  return pos;
}

// cos(2 pi n / d) and sin(2 pi n / d) at compile time: octant reduction, then the power series
constexpr double series(double x, bool sine) {
  double t = sine ? x : 1.0, s = t;
  for (int i = sine ? 2 : 1; i < 26; i += 2) {
    t *= -x * x / (double)(i * (i + 1));
    s += t;
  }
  return s;
}
constexpr double turn_cos(int n, int d) {
  if (n < 0) n = -n;
  n %= d;
  if (2 * n > d) n = d - n;
  if (4 * n > d) return -turn_cos(d - 2 * n, 2 * d);
  if (8 * n > d) return series(2.0 * M_PI * (double)(d - 4 * n) / (double)(4 * d), true);
  return series(2.0 * M_PI * (double)n / (double)d, false);
}
constexpr double turn_sin(int n, int d) { return turn_cos(4 * n - d, 4 * d); }

template <int R>
struct Roots {
  double c[R], s[R];
  constexpr Roots() : c(), s() {
    for (int j = 0; j < R; ++j) {
      c[j] = turn_cos(j, R);
      s[j] = turn_sin(j, R);
    }
  }
};

template <class T, int R, bool FWD>
struct GDftPow;  // R = 1, 2, 4, 8

// In-register DFT of length R: x_m <- sum_n x_n exp(-+ 2 pi i m n / R) (FWD: minus).  Odd primes in float32: term by
// term.  Outputs m and R - m use the same products but for signs, so they are formed together, and one pair
// after the other, or the products of all pairs are live at once (R = 13: 144).
template <class T, int R, bool FWD>
struct GDft {
  using C = Cx<T>;
  __device__ __forceinline__ static C output(const C (&x)[R], int m) {
    constexpr Roots<R> w{};
    C acc = x[0];
#pragma unroll
    for (int n = 1; n < R; ++n) {
      const int k = (m * n) % R;
      acc = gadd(acc, m == 0 ? x[n] : gmul(x[n], cmk<T>((T)w.c[k], FWD ? (T)-w.s[k] : (T)w.s[k])));
    }
    return acc;
  }
  __device__ __forceinline__ static void run(C (&x)[R]) {
    C y[R];
    y[0] = output(x, 0);
#pragma unroll
    for (int m = 1; m <= R / 2; ++m) {
      y[m] = output(x, m);
      y[R - m] = output(x, R - m);
      if (R >= 5) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int m = 0; m < R; ++m) x[m] = y[m];
  }
};
// In float64, whose rounding does not steer a clean, in the symmetric form: with a_j = x_j + x_{R-j} and
// b_j = x_j - x_{R-j}, outputs m and R-m share sum_j cos(2 pi m j / R) a_j and sum_j sin(2 pi m j / R) b_j, a
// quarter of the products.
template <int R, bool FWD>
struct GDft<double, R, FWD> {
  using T = double;
  using C = Cx<double>;
  __device__ __forceinline__ static void run(C (&x)[R]) {
    constexpr Roots<R> w{};
    constexpr int H = (R - 1) / 2;
    C a[H], b[H];
    C sum = x[0];
#pragma unroll
    for (int j = 0; j < H; ++j) {
      a[j] = gadd(x[j + 1], x[R - 1 - j]);
      b[j] = gsub(x[j + 1], x[R - 1 - j]);
      sum = gadd(sum, a[j]);
    }
    const C x0 = x[0];
    x[0] = sum;
#pragma unroll
    for (int m = 1; m <= H; ++m) {
      C u = x0, v = cmk<T>(w.s[m] * b[0].x, w.s[m] * b[0].y);
#pragma unroll
      for (int j = 0; j < H; ++j) {
        const T cc = w.c[(m * (j + 1)) % R];
        u = cmk<T>(fma(cc, a[j].x, u.x), fma(cc, a[j].y, u.y));
        if (j) {
          const T ss = w.s[(m * (j + 1)) % R];
          v = cmk<T>(fma(ss, b[j].x, v.x), fma(ss, b[j].y, v.y));
        }
      }
      const C iv = gmul_i<T, FWD>(v);
      x[m] = gadd(u, iv);
      x[R - m] = gsub(u, iv);
    }
  }
};
template <class T, bool FWD>
struct GDftPow<T, 1, FWD> {
  __device__ __forceinline__ static void run(Cx<T> (&)[1]) {}
};

template <class T, bool FWD>
struct GDftPow<T, 2, FWD> {
  using C = Cx<T>;
  __device__ __forceinline__ static void run(C (&x)[2]) {
    const C a = x[0], b = x[1];
    x[0] = gadd(a, b);
    x[1] = gsub(a, b);
  }
};

template <class T, bool FWD>
struct GDftPow<T, 4, FWD> {
  using C = Cx<T>;
  __device__ __forceinline__ static void run(C (&x)[4]) {
    const C s0 = gadd(x[0], x[2]), d0 = gsub(x[0], x[2]);
    const C s1 = gadd(x[1], x[3]), d1 = gmul_i<T, FWD>(gsub(x[1], x[3]));
    x[0] = gadd(s0, s1);
    x[2] = gsub(s0, s1);
    x[1] = gadd(d0, d1);
    x[3] = gsub(d0, d1);
  }
};

template <class T, bool FWD>
struct GDftPow<T, 8, FWD> {
  using C = Cx<T>;
  __device__ __forceinline__ static void run(C (&x)[8]) {
    C e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
    GDftPow<T, 4, FWD>::run(e);
    GDftPow<T, 4, FWD>::run(o);
    const T h = (T)0.70710678118654752440;  // cos(pi/4)
    // o_k * exp(-+ 2 pi i k / 8) for k = 0..3, those of 1 and 3 without their factor h
    const C u1 = FWD ? cmk<T>(o[1].x + o[1].y, o[1].y - o[1].x) : cmk<T>(o[1].x - o[1].y, o[1].y + o[1].x);
    const C t2 = gmul_i<T, FWD>(o[2]);
    const C u3 = FWD ? cmk<T>(o[3].y - o[3].x, -(o[3].x + o[3].y)) : cmk<T>(-(o[3].x + o[3].y), o[3].x - o[3].y);
    x[0] = gadd(e[0], o[0]);
    x[4] = gsub(e[0], o[0]);
    x[1] = cmk<T>(fma(h, u1.x, e[1].x), fma(h, u1.y, e[1].y));
    x[5] = cmk<T>(fma(-h, u1.x, e[1].x), fma(-h, u1.y, e[1].y));
    x[2] = gadd(e[2], t2);
    x[6] = gsub(e[2], t2);
    x[3] = cmk<T>(fma(h, u3.x, e[3].x), fma(h, u3.y, e[3].y));
    x[7] = cmk<T>(fma(-h, u3.x, e[3].x), fma(-h, u3.y, e[3].y));
  }
};

template <bool FWD, class T, int R>
__device__ __forceinline__ void dft(Cx<T> (&x)[R]) {
  if constexpr ((R & (R - 1)) == 0)
    GDftPow<T, R, FWD>::run(x);
  else
    GDft<T, R, FWD>::run(x);
}

// f(step_kind constants) for the run-time step kind
template <class F>
__device__ __forceinline__ void with_step(int kind, F&& f) {
  switch (kind) {
    case 0: f(std::integral_constant<int, 0>{}); break;
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 9: f(std::integral_constant<int, 9>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    default: f(std::integral_constant<int, 11>{}); break;
  }
}

// Twiddles of one butterfly of a step on sub-transforms of length Ls, butterfly index n within one.  tw: the
// plan's stage twiddles, exp(-2 pi i n k / Ls) of the stage of sub-transform length Ls at
// L - Ls + (k-1) M + n (M = Ls / radix), so that neighbouring butterflies read neighbouring entries.
template <class T, int R1, int R2>
struct StepTw {
  using C = Cx<T>;
  C w1[R1][R2];  // stage 1: element (k, j) at k M1 + j M2 + n
  C w2[R2];      // stage 2
  __device__ __forceinline__ void load(const C* __restrict__ tw, int L, int Ls, int n) {
    const int M1 = Ls / R1, M2 = M1 / R2;
    if (R2 > 1 || M1 > 1) {
      const C* t = tw + (L - Ls);
#pragma unroll
      for (int k = 1; k < R1; ++k)
#pragma unroll
        for (int j = 0; j < R2; ++j) w1[k][j] = t[(k - 1) * M1 + j * M2 + n];
    }
    if (R2 > 1 && M2 > 1) {
      const C* t = tw + (L - M1);
#pragma unroll
      for (int j = 1; j < R2; ++j) w2[j] = t[(j - 1) * M2 + n];
    }
  }
};

// The arithmetic of a step on the elements x[k * R2 + j] at k M1 + j M2.  Forward: stage 1 on the R1 elements of
// each j, then stage 2 on the R2 of each k, a DFT then twiddles each (decimation in frequency; the last stage of a
// transform has none).  Inverse: conjugate twiddles then the inverse DFT, the exact mirror.
template <class T, int R1, int R2, bool FWD>
__device__ __forceinline__ void step_math(Cx<T> (&x)[R1 * R2], const StepTw<T, R1, R2>& tw, bool tw1, bool tw2) {
  using C = Cx<T>;
  const auto stage1 = [&] {
#pragma unroll
    for (int j = 0; j < R2; ++j) {
      C y[R1];
#pragma unroll
      for (int k = 0; k < R1; ++k) y[k] = x[k * R2 + j];
      if (FWD) dft<true>(y);
      if (R2 > 1 || tw1) {
#pragma unroll
        for (int k = 1; k < R1; ++k) y[k] = gmul(y[k], FWD ? tw.w1[k][j] : gconj(tw.w1[k][j]));
      }
      if (!FWD) dft<false>(y);
#pragma unroll
      for (int k = 0; k < R1; ++k) x[k * R2 + j] = y[k];
    }
  };
  const auto stage2 = [&] {
    if constexpr (R2 > 1) {
#pragma unroll
      for (int k = 0; k < R1; ++k) {
        C y[R2];
#pragma unroll
        for (int j = 0; j < R2; ++j) y[j] = x[k * R2 + j];
        if (FWD) dft<true>(y);
        if (tw2) {
#pragma unroll
          for (int j = 1; j < R2; ++j) y[j] = gmul(y[j], FWD ? tw.w2[j] : gconj(tw.w2[j]));
        }
        if (!FWD) dft<false>(y);
#pragma unroll
        for (int j = 0; j < R2; ++j) x[k * R2 + j] = y[j];
      }
    }
  };
  if (FWD) {
    stage1();
    stage2();
  } else {
    stage2();
    stage1();
  }
}

// One step over a transform of length L, sub-transform length Ls, butterflies lt, lt + step, ...: elements from
// ld(i), results to st(i, v); a butterfly reads and writes the same elements, so a step can run in
// place.  SYNC: a barrier before the first element is read, behind the request of the first butterfly's
// twiddles.
template <class T, bool FWD, bool SYNC, class Ld, class St>
__device__ __forceinline__ void gstep(int kind, int L, int Ls, const Cx<T>* __restrict__ tw, int lt, int step, Ld ld,
                                      St st) {
  using C = Cx<T>;
  with_step(kind, [&](auto kc) {
    constexpr GStep S = step_kind(decltype(kc)::value);
    constexpr int R1 = S.r1, R2 = S.r2, R = R1 * R2;
    const int M1 = Ls / R1, M2 = M1 / R2;
    const int nbf = L / R;
    const float inv_m = 1.f / (float)M2;
    // b / M2: (b + 1/2) / M2 is at least 1/(2 M2) from a whole number, and the float product is off by less
    // than 2^-21 of it, which is at most 2^-8 / M2 for b < 2^13
    int b = lt;
    int blk = (int)(((float)b + 0.5f) * inv_m);
    int n = b - blk * M2;
    constexpr bool kAhead = R1 < 11;  // a large DFT holds its inputs and outputs: its twiddles come after it
    StepTw<T, R1, R2> w;
    if (kAhead && b < nbf) w.load(tw, L, Ls, n);
    if (SYNC) __syncthreads();
    while (b < nbf) {
      const int base = blk * Ls + n;
      C x[R];
#pragma unroll
      for (int k = 0; k < R1; ++k)
#pragma unroll
        for (int j = 0; j < R2; ++j) x[k * R2 + j] = ld(base + k * M1 + j * M2);
      if constexpr (kAhead) {
        step_math<T, R1, R2, FWD>(x, w, M1 > 1, M2 > 1);
      } else {
        if (FWD) dft<true>(x);
        __builtin_amdgcn_sched_barrier(0);
        if (M1 > 1) {
          const C* __restrict__ t = tw + (L - Ls) + n;
#pragma unroll
          for (int k = 1; k < R1; ++k) {
            const C v = t[(k - 1) * M1];
            x[k] = gmul(x[k], FWD ? v : gconj(v));
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (!FWD) dft<false>(x);
      }
#pragma unroll
      for (int k = 0; k < R1; ++k)
#pragma unroll
        for (int j = 0; j < R2; ++j) st(base + k * M1 + j * M2, x[k * R2 + j]);
      b += step;
      if (b < nbf) {
        blk = (int)(((float)b + 0.5f) * inv_m);
        n = b - blk * M2;
        if (kAhead) w.load(tw, L, Ls, n);
      }
    }
  });
}

// Tables of one frame side P, in one device allocation: stage twiddles of the P plan and of the P/2
// plan, the split factors exp(-2 pi i k / P) for k <= P/2, the digit reversal of the P/2 plan.
template <class T>
struct GTables {
  const Cx<T>* col;
  const Cx<T>* row;
  const Cx<T>* split;
  const uint16_t* perm;
};

template <class T, int NB>
struct GR2cBatch {
  const void* src[NB];
  Cx<T>* T1[NB];
  const int* pred[NB];
};
template <class T, int NB>
struct GColBatch {
  const Cx<T>* T1[NB];
  const Cx<T>* S[NB];
  Cx<T>* T2[NB];
  const int* pred[NB];
};
template <class T, int NB>
struct GC2rBatch {
  const Cx<T>* T2[NB];
  T* out[NB];
  const int* pred[NB];
};

// ---- pass 1: rows r2c.  Frame row fr of the job: the image row (off == 0, q x q image at the
// frame origin) or the PSF row of the centred, -P/2-rolled frame (off = q/2).  Output column-major:
// T1[k * ldT + fr], k in [0, P/2].
//
// A block transforms 2^lg neighbouring rows, element i of row g at LDS slot gpad(i) * 2^lg + g, lanes
// over rows first: T1 is written in runs of 2^lg values (single values of each column took most of
// the pass before), and the LDS accesses of the rows fall side by side.  The first stage reads the
// image, the split computes outputs k and L - k from one read of both.
// VEC: image rows of even length at aligned addresses, read two values at a time.
template <class T, class TIN, bool VEC, int NB>
__global__ __launch_bounds__(kGThreads, sizeof(T) == 4 ? 4 : 2) void k_g_r2c(GR2cBatch<T, NB> bt, GPlan pl, int P, int q, int off, int n_rows,
                                                     int ldT, int lg, GTables<T> tab) {
  using C = Cx<T>;
  const int jb = blockIdx.y;
  const int* pred = bt.pred[jb];
  if (pred && *pred == 0) return;
  const TIN* __restrict__ src = static_cast<const TIN*>(bt.src[jb]);
  C* __restrict__ T1 = bt.T1[jb];
  extern __shared__ unsigned char g_smem[];
  const int L = pl.L;
  const int g = threadIdx.x & ((1 << lg) - 1);
  const int lt = threadIdx.x >> lg;
  const int step = blockDim.x >> lg;
  const int fr = (int)(xcd_remap(blockIdx.x, gridDim.x) << lg) + g;
  C* sm = reinterpret_cast<C*>(g_smem) + g;
  const bool live = fr < n_rows;
  int a = fr + off;
  a = a >= P ? a - P : a;
  const bool row_ok = live && a < q;
  const TIN* row = src + (size_t)(row_ok ? a : 0) * q;
  const auto lds_ld = [&](int i) { return sm[gpad(i) << lg]; };
  const auto lds_st = [&](int i, C v) { sm[gpad(i) << lg] = v; };
  const auto image = [&](int e) {
    if constexpr (VEC) {
      struct alignas(2 * sizeof(TIN)) Two {
        TIN x, y;
      };
      const bool ok = row_ok && 2 * e < q;
      const Two v = reinterpret_cast<const Two*>(row)[ok ? e : 0];
      return ok ? cmk<T>((T)v.x, (T)v.y) : cmk<T>(0, 0);
    } else {
      int c0 = 2 * e + off, c1 = c0 + 1;
      c0 = c0 >= P ? c0 - P : c0;
      c1 = c1 >= P ? c1 - P : c1;
      const bool ok0 = row_ok && c0 < q, ok1 = row_ok && c1 < q;
      const T v0 = (T)row[ok0 ? c0 : 0], v1 = (T)row[ok1 ? c1 : 0];
      return cmk<T>(ok0 ? v0 : (T)0, ok1 ? v1 : (T)0);
    }
  };
  gstep<T, true, false>(pl.kind(0), L, L, tab.row, lt, step, image, lds_st);
  int Ls = L / pl.r(0);
  for (int i = 1; i < pl.ns; ++i) {
    gstep<T, true, true>(pl.kind(i), L, Ls, tab.row, lt, step, lds_ld, lds_st);
    Ls /= pl.r(i);
  }
  __syncthreads();
  if (!live) return;
  const auto split = [](C zk, C zl, C tw) {  // zl: conj z_{L-k}
    const C e = gscale(gadd(zk, zl), (T)0.5);
    const C dd = gscale(gsub(zk, zl), (T)0.5);
    const C o = cmk<T>(dd.y, -dd.x);  // (zk - conj z_{L-k}) / (2i)
    return gadd(e, gmul(tw, o));
  };
  for (int k = lt; 2 * k <= L; k += step) {
    const C zk = lds_ld(tab.perm[k]);
    const C zl = gconj(lds_ld(tab.perm[k == 0 ? 0 : L - k]));
    T1[(size_t)k * ldT + fr] = split(zk, zl, tab.split[k]);
    if (2 * k < L) T1[(size_t)(L - k) * ldT + fr] = split(gconj(zl), gconj(zk), tab.split[L - k]);
  }
}

// ---- pass 2: per frequency column k in [0, P/2]: the n_in stored rows (zero beyond) -> forward
// P-point FFT.  SPEC: store the spectrum column.  Otherwise multiply by the PSF column, inverse
// FFT, store the first n_out rows: T2[k * n_out + i].
//
// The first step reads the column, the last inverse step stores it; between them the last forward
// step, the product and the first inverse step work on the same r elements and stay in registers.
// The spectrum is stored as they read it: element k of butterfly b at k * (P/r) + b.
template <class T, bool SPEC, int NB>
__global__ __launch_bounds__(kGThreads, sizeof(T) == 4 ? 4 : 2) void k_g_cols(GColBatch<T, NB> bt, GPlan pl, int n_in, int n_out, int G,
                                                      GTables<T> tab) {
  using C = Cx<T>;
  const int jb = blockIdx.y;
  const int* pred = bt.pred[jb];
  if (pred && *pred == 0) return;
  extern __shared__ unsigned char g_smem[];
  const int P = pl.L;
  const int ncols = P / 2 + 1;
  const int step = blockDim.x / G;
  const int g = threadIdx.x / step;
  const int lt = threadIdx.x - g * step;
  const int k = blockIdx.x * G + g;
  const bool live = k < ncols;
  C* sm = reinterpret_cast<C*>(g_smem) + g * gspan(P);
  const C* __restrict__ col = bt.T1[jb] + (size_t)(live ? k : 0) * n_in;
  const auto lds_ld = [&](int i) { return sm[gpad(i)]; };
  const auto lds_st = [&](int i, C v) { sm[gpad(i)] = v; };
  const auto column = [&](int i) {
    const C v = col[i < n_in ? i : 0];
    return i < n_in ? v : cmk<T>(0, 0);
  };
  gstep<T, true, false>(pl.kind(0), P, P, tab.col, lt, step, column, lds_st);
  int Ls = P / pl.r(0);
  const int last = pl.ns - 1;
  for (int i = 1; i < last; ++i) {
    gstep<T, true, true>(pl.kind(i), P, Ls, tab.col, lt, step, lds_ld, lds_st);
    Ls /= pl.r(i);
  }
  C* __restrict__ out = bt.T2[jb] + (size_t)(live ? k : 0) * (SPEC ? P : n_out);
  const C* __restrict__ S = SPEC ? nullptr : bt.S[jb] + (size_t)(live ? k : 0) * P;
  with_step(pl.kind(last), [&](auto kc) {
    constexpr GStep K = step_kind(decltype(kc)::value);
    constexpr int R1 = K.r1, R2 = K.r2, R = R1 * R2;
    const int nbf = P / R;
    int b = lt;
    StepTw<T, R1, R2> w;
    if (R2 > 1) w.load(tab.col, P, R, 0);
    constexpr bool kAhead = R1 < 11;
    C s[R];
    if (!SPEC && kAhead && b < nbf) {
#pragma unroll
      for (int m = 0; m < R; ++m) s[m] = S[m * nbf + b];
    }
    __syncthreads();
    while (b < nbf) {
      C x[R];
#pragma unroll
      for (int m = 0; m < R; ++m) x[m] = lds_ld(b * R + m);
      step_math<T, R1, R2, true>(x, w, false, false);
      if (SPEC) {
        if (live) {
#pragma unroll
          for (int m = 0; m < R; ++m) out[m * nbf + b] = x[m];
        }
      } else {
        if (!kAhead) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int m = 0; m < R; ++m) s[m] = S[m * nbf + b];
        }
#pragma unroll
        for (int m = 0; m < R; ++m) x[m] = gmul(x[m], s[m]);
        if (!kAhead) __builtin_amdgcn_sched_barrier(0);
        step_math<T, R1, R2, false>(x, w, false, false);
#pragma unroll
        for (int m = 0; m < R; ++m) lds_st(b * R + m, x[m]);
      }
      b += step;
      if (!SPEC && kAhead && b < nbf) {
#pragma unroll
        for (int m = 0; m < R; ++m) s[m] = S[m * nbf + b];
      }
    }
  });
  if (SPEC) return;
  for (int i = last - 1; i > 0; --i) {
    Ls *= pl.r(i);
    gstep<T, false, true>(pl.kind(i), P, Ls, tab.col, lt, step, lds_ld, lds_st);
  }
  const auto kept = [&](int i, C v) {
    if (live && i < n_out) out[i] = v;
  };
  gstep<T, false, true>(pl.kind(0), P, P, tab.col, lt, step, lds_ld, kept);
}

// ---- pass 3: per kept row r: Hermitian half spectrum T2[k * ldT + r], k in [0, P/2] -> the
// P/2-point complex sequence whose inverse FFT interleaves the even and odd output samples, scaled
// by 1/P^2; the first n columns are stored.  Rows share a block as in pass 1; frequencies k and L - k are
// read once for both their elements, and the last stage stores the image.
// VEC: output rows of even length at aligned addresses.
template <class T, bool VEC, int NB>
__global__ __launch_bounds__(kGThreads, sizeof(T) == 4 ? 4 : 2) void k_g_c2r(GC2rBatch<T, NB> bt, GPlan pl, int n, int ldT, int lg, T scale,
                                                     GTables<T> tab) {
  using C = Cx<T>;
  const int jb = blockIdx.y;
  const int* pred = bt.pred[jb];
  if (pred && *pred == 0) return;
  extern __shared__ unsigned char g_smem[];
  const int L = pl.L;
  const int g = threadIdx.x & ((1 << lg) - 1);
  const int lt = threadIdx.x >> lg;
  const int step = blockDim.x >> lg;
  const int r = (int)(xcd_remap(blockIdx.x, gridDim.x) << lg) + g;
  const bool live = r < n;
  C* sm = reinterpret_cast<C*>(g_smem) + g;
  const C* __restrict__ T2 = bt.T2[jb] + (live ? r : 0);
  const auto lds_ld = [&](int i) { return sm[gpad(i) << lg]; };
  const auto lds_st = [&](int i, C v) { sm[gpad(i) << lg] = v; };
  const auto merge = [](C xk, C xl, C tw) {  // xl: conj X_{L-k}
    const C d = gmul(gsub(xk, xl), gconj(tw));  // (X_k - conj X_{L-k}) exp(+2 pi i k / P)
    return gadd(gadd(xk, xl), cmk<T>(-d.y, d.x));
  };
  for (int k = lt; 2 * k <= L; k += step) {
    const C xk = T2[(size_t)k * ldT];
    const C xl = gconj(T2[(size_t)(L - k) * ldT]);
    lds_st(tab.perm[k], merge(xk, xl, tab.split[k]));
    if (k > 0 && 2 * k < L) lds_st(tab.perm[L - k], merge(gconj(xl), gconj(xk), tab.split[L - k]));
  }
  int Ls = 1;
  for (int i = pl.ns - 1; i > 0; --i) {
    Ls *= pl.r(i);
    gstep<T, false, true>(pl.kind(i), L, Ls, tab.row, lt, step, lds_ld, lds_st);
  }
  T* __restrict__ out = bt.out[jb] + (size_t)(live ? r : 0) * n;
  const auto image = [&](int e, C v) {
    if constexpr (VEC) {
      if (live && 2 * e < n) reinterpret_cast<C*>(out)[e] = gscale(v, scale);
    } else {
      if (live && 2 * e < n) out[2 * e] = v.x * scale;
      if (live && 2 * e + 1 < n) out[2 * e + 1] = v.y * scale;
    }
  };
  gstep<T, false, true>(pl.kind(0), L, L, tab.row, lt, step, lds_ld, image);
}

// ---- host side --------------------------------------------------------------------------------
// The plan of length L: its stages are radix 8 while the length allows, a 4 or 2 for the rest of the power of
// two, then the odd primes in order (which fixes every rounding); neighbouring stages are taken together where a
// step kind has them, with the fewest steps, at least min_steps (each is a pass through LDS and a barrier).
bool make_gplan(int L, int min_steps, GPlan* p) {
  constexpr int kMostStages = 16;
  int r[kMostStages], n = 0, m = L;
  for (int f : {8, 4, 2, 3, 5, 7, 11, 13})
    while (m % f == 0 && n < kMostStages) {
      r[n++] = f;
      m /= f;
      if (f == 4 || f == 2) break;  // at most one of each is left by the eights
    }
  if (m != 1 || n == 0) return false;
  const auto kind_of = [&](int i, int count) {  // the step of `count` stages from stage i on, or -1
    for (int k = 0; k < kStepKinds; ++k)
      if (step_kind(k).r1 == r[i] && step_kind(k).r2 == (count == 2 ? r[i + 1] : 1)) return k;
    return -1;
  };
  int steps[kMostStages + 1], take[kMostStages];  // from stage i on: the fewest steps, the stages of the first of them
  steps[n] = 0;
  for (int i = n - 1; i >= 0; --i) {
    steps[i] = 1 + steps[i + 1];
    take[i] = 1;
    const bool two = i + 1 < n && kind_of(i, 2) >= 0 && !(i == 0 && n == 2 && min_steps == 2);
    if (two && 1 + steps[i + 2] < steps[i]) {
      steps[i] = 1 + steps[i + 2];
      take[i] = 2;
    }
  }
  if (steps[0] > kMaxSteps || steps[0] < min_steps) return false;
  p->L = L;
  p->ns = 0;
  p->code = 0;
  for (int i = 0; i < n; i += take[i]) p->code |= (uint32_t)kind_of(i, take[i]) << (4 * p->ns++);
  return true;
}
bool row_plan(int p, GPlan* pl) { return make_gplan(p / 2, 1, pl); }
bool col_plan(int p, GPlan* pl) { return make_gplan(p, 2, pl); }

struct Shape {
  int groups_log2;  // log2 of the transforms per block
  int threads;
  size_t lds;
};

// Row passes: four rows a block (32-byte runs of the float32 intermediate), fewer where they do not fit
// half a CU's LDS, and a thread per butterfly of radix 5.  One, two and eight rows a block measured 3 us
// slower to 1 us faster, 2 us either way and 3 us slower per convolution at frames of 500 to 3000, 33, 0 and 15 us
// slower at 6000; radix 8 for the threads 1 us slower up to frames of 1200.
Shape row_shape(int L, size_t elem) {
  int lg = 2;
  while (lg > 0 && ((size_t)gspan(L) * elem << lg) > 80 * 1024) --lg;
  const int want = (int)(((long)L << lg) / 5);
  const int threads = std::max(64, std::min(kGThreads, ceil_div(want, 64) * 64));
  return {lg, threads, (size_t)gspan(L) * elem << lg};
}

// Column pass: one column a block, a thread per butterfly of radix 5 up to 256 threads: the registers hold
// 16 waves of a CU in float32 (8 in float64), in four blocks (two) of four waves each, as long as those fit the LDS (512
// threads: 53 against 46 us at a frame of 2200, 81 against 70 us at 3600); one large block where they do not.
// Short columns share a wave.
Shape col_shape(int P, size_t elem) {
  if (P <= 160) {
    const int step = P <= 80 ? 16 : 32;
    return {step == 16 ? 2 : 1, 64, (size_t)gspan(P) * elem << (step == 16 ? 2 : 1)};
  }
  const int most = gspan(P) <= 5 * 1024 ? 256 : kGThreads;
  return {0, std::min(most, ceil_div(P / 5, 64) * 64), (size_t)gspan(P) * elem};
}

struct TwKey {
  int dev, p, bytes;
  bool operator<(const TwKey& o) const {
    return dev != o.dev ? dev < o.dev : (p != o.p ? p < o.p : bytes < o.bytes);
  }
};
std::mutex g_gtw_mu;
std::map<TwKey, void*> g_gtw;

// stage twiddles of a plan, laid out as StepTw reads them, from w[k] = exp(-2 pi i k / P)
template <class C>
void stage_twiddles(const GPlan& pl, const std::vector<C>& w, C* out) {
  const int P = (int)w.size();
  int Ls = pl.L;
  for (int i = 0; i < pl.ns; ++i) {
    const GStep st = step_kind(pl.kind(i));
    for (int r : {st.r1, st.r2}) {
      const int M = Ls / r, tstep = P / Ls;
      for (int k = 1; k < r; ++k)
        for (int n = 0; n < M; ++n) out[pl.L - Ls + (k - 1) * M + n] = w[(size_t)n * k * tstep];
      Ls = M;
    }
  }
}

// the tables of frame side p in type T (computed in float64), one allocation per device and p
template <class T>
GTables<T> g_tables(int p) {
  using C = Cx<T>;
  const int L = p / 2, n_split = L + 1;
  int dev = 0;
  PMS_HIP(hipGetDevice(&dev));
  const TwKey key{dev, p, (int)sizeof(T)};
  const auto view = [&](void* d) {
    const C* c = static_cast<const C*>(d);
    return GTables<T>{c, c + p, c + p + L, reinterpret_cast<const uint16_t*>(c + p + L + n_split)};
  };
  std::lock_guard<std::mutex> lk(g_gtw_mu);
  auto it = g_gtw.find(key);
  if (it != g_gtw.end()) return view(it->second);
  std::vector<C> w(p);
  for (int k = 0; k < p; ++k) {
    const double a = -2.0 * M_PI * (double)k / (double)p;
    w[k].x = (T)std::cos(a);
    w[k].y = (T)std::sin(a);
  }
  const size_t bytes = sizeof(C) * (size_t)(p + L + n_split) + sizeof(uint16_t) * (size_t)L;
  std::vector<unsigned char> h(bytes);
  C* c = reinterpret_cast<C*>(h.data());
  GPlan pl;
  col_plan(p, &pl);
  stage_twiddles(pl, w, c);
  row_plan(p, &pl);
  stage_twiddles(pl, w, c + p);
  std::copy(w.begin(), w.begin() + n_split, c + p + L);
  uint16_t* perm = reinterpret_cast<uint16_t*>(c + p + L + n_split);
  for (int k = 0; k < L; ++k) perm[k] = (uint16_t)gperm(pl, k);
  void* d = nullptr;
  PMS_HIP(hipMalloc(&d, bytes));
  PMS_HIP(hipMemcpy(d, h.data(), bytes, hipMemcpyHostToDevice));
  g_gtw.emplace(key, d);
  return view(d);
}

template <class T>
void set_g_attrs() {
  static std::once_flag once;
  std::call_once(once, [] {
    const int lds_max = 160 * 1024;
    auto allow = [&](const void* k) {
      (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
    };
    allow((const void*)k_g_r2c<T, float, false, 1>);
    if constexpr (sizeof(T) == 8) allow((const void*)k_g_r2c<T, double, false, 1>);
    allow((const void*)k_g_r2c<T, T, true, 1>);
    allow((const void*)k_g_r2c<T, T, false, kMaxBatch>);
    allow((const void*)k_g_r2c<T, T, true, kMaxBatch>);
    allow((const void*)k_g_cols<T, true, 1>);
    allow((const void*)k_g_cols<T, false, 1>);
    allow((const void*)k_g_cols<T, false, kMaxBatch>);
    allow((const void*)k_g_c2r<T, false, 1>);
    allow((const void*)k_g_c2r<T, true, 1>);
    allow((const void*)k_g_c2r<T, false, kMaxBatch>);
    allow((const void*)k_g_c2r<T, true, kMaxBatch>);
    (void)hipGetLastError();
  });
}

// Frames whose transforms there are kernels for: powers of two run on their own (fft_pow2.h), whatever
// the steps below could make of them (4 and 8 are a single stage, which a column plan cannot be).
bool has_kernels(int p) {
  GPlan pl;
  return is_pow2(p) || (col_plan(p, &pl) && row_plan(p, &pl));
}

template <class T>
void check_g_frame(int p) {
  PMS_REQUIRE(p >= 4 && p % 2 == 0, "FFT frame side must be even and >= 4, got " + std::to_string(p));
  PMS_REQUIRE(p <= gfft_max_frame(sizeof(T)),
              "FFT frame side " + std::to_string(p) + " exceeds the " + std::to_string(gfft_max_frame(sizeof(T))) +
                  " that one LDS transform holds in " + (sizeof(T) == 8 ? "float64" : "float32"));
  PMS_REQUIRE(has_kernels(p), "FFT frame side " + std::to_string(p) + " has a prime factor above 13");
}

template <class T, class TIN, bool VEC, int NB>
void launch_r2c(const GR2cBatch<T, NB>& bt, int nb, int p, int q, int off, int n_rows, int ldT,
                const GTables<T>& tab, hipStream_t st) {
  GPlan pl;
  row_plan(p, &pl);
  const Shape s = row_shape(p / 2, sizeof(Cx<T>));
  hipLaunchKernelGGL((k_g_r2c<T, TIN, VEC, NB>), dim3(ceil_div(n_rows, 1 << s.groups_log2), nb), dim3(s.threads), s.lds,
                     st, bt, pl, p, q, off, n_rows, ldT, s.groups_log2, tab);
  PMS_LAUNCH_CHECK();
}

template <class T, bool SPEC, int NB>
void launch_cols(const GColBatch<T, NB>& bt, int nb, int p, int n_in, int n_out, const GTables<T>& tab,
                 hipStream_t st) {
  GPlan pl;
  col_plan(p, &pl);
  const Shape s = col_shape(p, sizeof(Cx<T>));
  const int G = 1 << s.groups_log2;
  hipLaunchKernelGGL((k_g_cols<T, SPEC, NB>), dim3(ceil_div(p / 2 + 1, G), nb), dim3(s.threads), s.lds, st, bt, pl, n_in,
                     n_out, G, tab);
  PMS_LAUNCH_CHECK();
}

template <class T, bool VEC, int NB>
void launch_c2r(const GC2rBatch<T, NB>& bt, int nb, int p, int n, int ldT, const GTables<T>& tab, hipStream_t st) {
  GPlan pl;
  row_plan(p, &pl);
  const Shape s = row_shape(p / 2, sizeof(Cx<T>));
  const T scale = (T)(1.0 / ((double)p * (double)p));
  hipLaunchKernelGGL((k_g_c2r<T, VEC, NB>), dim3(ceil_div(n, 1 << s.groups_log2), nb), dim3(s.threads), s.lds, st, bt,
                     pl, n, ldT, s.groups_log2, scale, tab);
  PMS_LAUNCH_CHECK();
}

}  // namespace

int gfft_max_frame(size_t real_bytes) { return real_bytes == 8 ? 8192 : 16384; }

bool gfft_frame_ok(int p, size_t real_bytes) {
  return p >= 4 && p % 2 == 0 && p <= gfft_max_frame(real_bytes) && has_kernels(p);
}

int gfft_perm(int k, int p) {
  GPlan pl;
  PMS_REQUIRE(col_plan(p, &pl), "FFT frame side " + std::to_string(p) + " has a prime factor above 13");
  const int pos = gperm(pl, k), r = pl.r(pl.ns - 1);  // element pos % r of the last stage's butterfly pos / r
  return pos % r * (p / r) + pos / r;
}

template <class T, class TIN>
void gfft_psf_spectrum(const TIN* psf, int q, int p, Cx<T>* spec, Cx<T>* work,
                       hipStream_t st) {
  check_g_frame<T>(p);
  PMS_REQUIRE(q >= 1 && q <= p, "PSF larger than the FFT frame");
  if constexpr (sizeof(T) == 8) {
    if (is_pow2(p)) {
      pow2_psf_spectrum_f64(psf, q, p, spec, work, st);
      return;
    }
  }
  set_g_attrs<T>();
  const GTables<T> tab = g_tables<T>(p);
  GR2cBatch<T, 1> rb{};
  rb.src[0] = psf;
  rb.T1[0] = work;
  launch_r2c<T, TIN, false>(rb, 1, p, q, q / 2, p, p, tab, st);
  GColBatch<T, 1> cb{};
  cb.T1[0] = work;
  cb.T2[0] = spec;
  launch_cols<T, true>(cb, 1, p, p, p, tab, st);
}

namespace {
template <class T, int NB>
void gfft_conv_jobs(const GConvJob<T>* jobs, int nb, int n, int p, const GTables<T>& tab, hipStream_t st) {
  GR2cBatch<T, NB> rb{};
  GColBatch<T, NB> cb{};
  GC2rBatch<T, NB> ob{};
  bool vec_in = n % 2 == 0, vec_out = n % 2 == 0;  // two values at a time where every row starts aligned for it
  for (int k = 0; k < nb; ++k) {
    const GConvJob<T>& j = jobs[k];
    PMS_REQUIRE(j.in && j.spec && j.out && j.work, "fft_conv: NULL buffer");
    auto* T1 = j.work;
    auto* T2 = j.work + (size_t)(p / 2 + 1) * n;
    rb.src[k] = j.in;
    rb.T1[k] = T1;
    rb.pred[k] = j.pred;
    cb.T1[k] = T1;
    cb.S[k] = j.spec;
    cb.T2[k] = T2;
    cb.pred[k] = j.pred;
    ob.T2[k] = T2;
    ob.out[k] = j.out;
    ob.pred[k] = j.pred;
    vec_in = vec_in && reinterpret_cast<uintptr_t>(j.in) % sizeof(Cx<T>) == 0;
    vec_out = vec_out && reinterpret_cast<uintptr_t>(j.out) % sizeof(Cx<T>) == 0;
  }
  if (vec_in)
    launch_r2c<T, T, true>(rb, nb, p, n, 0, n, n, tab, st);
  else
    launch_r2c<T, T, false>(rb, nb, p, n, 0, n, n, tab, st);
  launch_cols<T, false>(cb, nb, p, n, n, tab, st);
  if (vec_out)
    launch_c2r<T, true>(ob, nb, p, n, n, tab, st);
  else
    launch_c2r<T, false>(ob, nb, p, n, n, tab, st);
}
}  // namespace

template <class T>
void gfft_conv_batch(const GConvJob<T>* jobs, int count, int n, int p, hipStream_t st) {
  check_g_frame<T>(p);
  PMS_REQUIRE(p == n || p == 2 * n, "fft_conv: frame must be N (circular) or 2N (linear)");
  if constexpr (sizeof(T) == 8) {
    if (is_pow2(p)) {
      pow2_conv_batch_f64(jobs, count, n, p, st);
      return;
    }
  }
  set_g_attrs<T>();
  const GTables<T> tab = g_tables<T>(p);
  for (int j0 = 0; j0 < count; j0 += kMaxBatch) {
    const int nb = std::min(kMaxBatch, count - j0);
    if (nb == 1)
      gfft_conv_jobs<T, 1>(jobs + j0, nb, n, p, tab, st);
    else
      gfft_conv_jobs<T, kMaxBatch>(jobs + j0, nb, n, p, tab, st);
  }
}

template void gfft_psf_spectrum<float, float>(const float*, int, int, Cx<float>*, Cx<float>*, hipStream_t);
template void gfft_psf_spectrum<double, float>(const float*, int, int, Cx<double>*, Cx<double>*, hipStream_t);
template void gfft_psf_spectrum<double, double>(const double*, int, int, Cx<double>*, Cx<double>*, hipStream_t);
template void gfft_conv_batch<float>(const GConvJob<float>*, int, int, int, hipStream_t);
template void gfft_conv_batch<double>(const GConvJob<double>*, int, int, int, hipStream_t);

}  // namespace pms
