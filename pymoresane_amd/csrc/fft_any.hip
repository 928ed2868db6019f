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
// spectrum is stored in the order in which the column pass multiplies by it.  The radices (2 to 16)
// are chosen on the host per length, the stages are compiled per radix.  Stage twiddles, split factors
// and the row transforms' digit reversal come from tables per frame side and type, computed on the host in float64.
//
// What bounds the passes is the chain of each block: its loads, one LDS exchange and barrier per stage, its
// stores.  So stages are few (radices to 16), the first and last ones work on global memory, twiddles and
// the PSF column are requested ahead of the barriers, nothing divides by a run-time number, and the
// blocks are small enough for 16 waves a CU.  Convolution of a 1000^2 image on a frame of 2000: rows r2c 10 us, columns
// 18 us, rows c2r 9 us (27 + 37 + 27 us with stages up to radix 8, a division per butterfly, run-time digit
// reversal and two rows a block); frames of 132 / 800 / 3000 / 6000: 39 / 50 / 180 / 718 -> 16 / 21 / 68 / 232 us.
// Error against 64 bits 3.0e-7 in the mean (3.1e-7 before).
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

constexpr int kMaxStages = 8;
constexpr int kMaxRadix = 16;

// Radix plan of one transform length: stage i (decimation-in-frequency order) has radix r(i) and
// works on sub-transforms of length Ls_i = L / (r(0) ... r(i-1)).  Four bits a radix (minus one):
// kernel arguments stay small.
struct GPlan {
  int L;
  int ns;
  uint32_t code;
  __host__ __device__ __forceinline__ int r(int i) const { return (int)((code >> (4 * i)) & 15u) + 1; }
};

// Position of frequency k in the digit-reversed output of the forward transform:
// k = d0 + r0 (d1 + r1 (d2 + ...)), position = d0 L/r0 + d1 L/(r0 r1) + ...
int gperm(const GPlan& p, int k) {
  int pos = 0, span = p.L;
  for (int i = 0; i < p.ns; ++i) {
    const int r = p.r(i);
    span /= r;
    const int q = k / r;
    pos += (k - q * r) * span;
    k = q;
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

// In-register DFT of length R: x_m <- sum_n x_n exp(-+ 2 pi i m n / R) (FWD: minus).  Odd primes in
// the symmetric form: with a_j = x_j + x_{R-j} and b_j = x_j - x_{R-j}, outputs m and R-m share
// sum_j cos(2 pi m j / R) a_j and sum_j sin(2 pi m j / R) b_j, a quarter of the direct form's products.
template <class T, int R, bool FWD>
struct GDft {
  using C = Cx<T>;
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
      C u = x0, v = cmk<T>((T)w.s[m] * b[0].x, (T)w.s[m] * b[0].y);
#pragma unroll
      for (int j = 0; j < H; ++j) {
        const T cc = (T)w.c[(m * (j + 1)) % R];
        u = cmk<T>(fma(cc, a[j].x, u.x), fma(cc, a[j].y, u.y));
        if (j) {
          const T ss = (T)w.s[(m * (j + 1)) % R];
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
struct GDft<T, 2, FWD> {
  using C = Cx<T>;
  __device__ __forceinline__ static void run(C (&x)[2]) {
    const C a = x[0], b = x[1];
    x[0] = gadd(a, b);
    x[1] = gsub(a, b);
  }
};

template <class T, bool FWD>
struct GDft<T, 4, FWD> {
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
struct GDft<T, 8, FWD> {
  using C = Cx<T>;
  __device__ __forceinline__ static void run(C (&x)[8]) {
    C e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
    GDft<T, 4, FWD>::run(e);
    GDft<T, 4, FWD>::run(o);
    const T h = (T)0.70710678118654752440;  // cos(pi/4)
    // o_k * exp(-+ 2 pi i k / 8) for k = 0..3
    const C t1 = FWD ? cmk<T>(h * (o[1].x + o[1].y), h * (o[1].y - o[1].x))
                     : cmk<T>(h * (o[1].x - o[1].y), h * (o[1].y + o[1].x));
    const C t2 = gmul_i<T, FWD>(o[2]);
    const C t3 = FWD ? cmk<T>(h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y))
                     : cmk<T>(-h * (o[3].x + o[3].y), h * (o[3].x - o[3].y));
    x[0] = gadd(e[0], o[0]);
    x[4] = gsub(e[0], o[0]);
    x[1] = gadd(e[1], t1);
    x[5] = gsub(e[1], t1);
    x[2] = gadd(e[2], t2);
    x[6] = gsub(e[2], t2);
    x[3] = gadd(e[3], t3);
    x[7] = gsub(e[3], t3);
  }
};

// Composite length A * B: B transforms of length A, the products with exp(-+ 2 pi i b m / AB), A
// transforms of length B.
template <class T, int A, int B, bool FWD>
struct GDft2 {
  using C = Cx<T>;
  __device__ __forceinline__ static void run(C (&x)[A * B]) {
    constexpr Roots<A * B> w{};
    C y[B][A];
#pragma unroll
    for (int b = 0; b < B; ++b) {
#pragma unroll
      for (int a = 0; a < A; ++a) y[b][a] = x[B * a + b];
      GDft<T, A, FWD>::run(y[b]);
      if (b) {
#pragma unroll
        for (int m = 1; m < A; ++m) {
          if (4 * b * m == A * B)
            y[b][m] = gmul_i<T, FWD>(y[b][m]);
          else
            y[b][m] = gmul(y[b][m], cmk<T>((T)w.c[b * m], FWD ? (T)-w.s[b * m] : (T)w.s[b * m]));
        }
      }
    }
#pragma unroll
    for (int m = 0; m < A; ++m) {
      C z[B];
#pragma unroll
      for (int b = 0; b < B; ++b) z[b] = y[b][m];
      GDft<T, B, FWD>::run(z);
#pragma unroll
      for (int q = 0; q < B; ++q) x[m + A * q] = z[q];
    }
  }
};

// The same for coprime A and B without the products (Good-Thomas): input (B a + A b) mod AB, output the m
// with m = m_A mod A and m = m_B mod B.
template <class T, int A, int B, bool FWD>
struct GDftCoprime {
  using C = Cx<T>;
  __device__ __forceinline__ static constexpr int out(int ma, int mb) {
    int m = ma;
    while (m % B != mb) m += A;
    return m;
  }
  __device__ __forceinline__ static void run(C (&x)[A * B]) {
    C y[B][A];
#pragma unroll
    for (int b = 0; b < B; ++b) {
#pragma unroll
      for (int a = 0; a < A; ++a) y[b][a] = x[(B * a + A * b) % (A * B)];
      GDft<T, A, FWD>::run(y[b]);
    }
#pragma unroll
    for (int m = 0; m < A; ++m) {
      C z[B];
#pragma unroll
      for (int b = 0; b < B; ++b) z[b] = y[b][m];
      GDft<T, B, FWD>::run(z);
#pragma unroll
      for (int q = 0; q < B; ++q) x[out(m, q)] = z[q];
    }
  }
};
template <class T, bool FWD>
struct GDft<T, 6, FWD> : GDftCoprime<T, 2, 3, FWD> {};
template <class T, bool FWD>
struct GDft<T, 9, FWD> : GDft2<T, 3, 3, FWD> {};
template <class T, bool FWD>
struct GDft<T, 10, FWD> : GDftCoprime<T, 2, 5, FWD> {};
template <class T, bool FWD>
struct GDft<T, 12, FWD> : GDftCoprime<T, 4, 3, FWD> {};
template <class T, bool FWD>
struct GDft<T, 14, FWD> : GDftCoprime<T, 2, 7, FWD> {};
template <class T, bool FWD>
struct GDft<T, 15, FWD> : GDftCoprime<T, 3, 5, FWD> {};
template <class T, bool FWD>
struct GDft<T, 16, FWD> : GDft2<T, 4, 4, FWD> {};

// f(std::integral_constant<int, R>) for the run-time radix r, 2 to 16
template <class F>
__device__ __forceinline__ void with_radix(int r, F&& f) {
  switch (r) {
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 9: f(std::integral_constant<int, 9>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    case 11: f(std::integral_constant<int, 11>{}); break;
    case 12: f(std::integral_constant<int, 12>{}); break;
    case 13: f(std::integral_constant<int, 13>{}); break;
    case 14: f(std::integral_constant<int, 14>{}); break;
    case 15: f(std::integral_constant<int, 15>{}); break;
    default: f(std::integral_constant<int, 16>{}); break;
  }
}

// One stage of radix r over a transform of length L, sub-transform length Ls (M = Ls/r), butterflies
// lt, lt + step, ...: elements from ld(i), results to st(i, v); a butterfly reads and writes the
// same r elements, so a stage can run in place.  Forward: DFT then twiddles (decimation in
// frequency); inverse: conjugate twiddles then the inverse DFT, the exact mirror.  tw: the plan's
// stage twiddles, exp(-2 pi i n k / Ls) at L - Ls + (k-1) M + n, so that neighbouring butterflies read
// neighbouring entries.  SYNC: a barrier before the first element is read, behind the request of the
// first butterfly's twiddles.
template <class T, bool FWD, bool SYNC, class Ld, class St>
__device__ __forceinline__ void gstage(int r, int L, int Ls, const Cx<T>* __restrict__ tw, int lt, int step, Ld ld,
                                       St st) {
  using C = Cx<T>;
  with_radix(r, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    const int M = Ls / R;
    const int nbf = L / R;
    const float inv_m = 1.f / (float)M;
    const C* __restrict__ ts = tw + (L - Ls);
    // b / M: (b + 1/2) / M is at least 1/(2M) from a whole number, and the float product is off by less
    // than 2^-21 of it, which is at most 2^-8 / M for b < 2^13
    int b = lt;
    int blk = (int)(((float)b + 0.5f) * inv_m);
    int n = b - blk * M;
    C w[R];
    if (M > 1 && b < nbf) {
#pragma unroll
      for (int k = 1; k < R; ++k) w[k] = ts[(k - 1) * M + n];
    }
    if (SYNC) __syncthreads();
    while (b < nbf) {
      const int base = blk * Ls + n;
      C x[R];
#pragma unroll
      for (int k = 0; k < R; ++k) x[k] = ld(base + k * M);
      if (FWD) GDft<T, R, true>::run(x);
      if (M > 1) {
#pragma unroll
        for (int k = 1; k < R; ++k) x[k] = gmul(x[k], FWD ? w[k] : gconj(w[k]));
      }
      if (!FWD) GDft<T, R, false>::run(x);
#pragma unroll
      for (int k = 0; k < R; ++k) st(base + k * M, x[k]);
      b += step;
      if (b < nbf) {
        blk = (int)(((float)b + 0.5f) * inv_m);
        n = b - blk * M;
        if (M > 1) {
#pragma unroll
          for (int k = 1; k < R; ++k) w[k] = ts[(k - 1) * M + n];
        }
      }
    }
  });
}

// Tables of one frame side P, in one device allocation: stage twiddles of the P plan and of the P/2
// plan, the split factors exp(-2 pi i k / P) for k <= P/4, the digit reversal of the P/2 plan.
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
__global__ __launch_bounds__(kGThreads) void k_g_r2c(GR2cBatch<T, NB> bt, GPlan pl, int P, int q, int off, int n_rows,
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
  gstage<T, true, false>(pl.r(0), L, L, tab.row, lt, step, image, lds_st);
  int Ls = L / pl.r(0);
  for (int i = 1; i < pl.ns; ++i) {
    gstage<T, true, true>(pl.r(i), L, Ls, tab.row, lt, step, lds_ld, lds_st);
    Ls /= pl.r(i);
  }
  __syncthreads();
  if (!live) return;
  for (int k = lt; 2 * k <= L; k += step) {
    const C zk = lds_ld(tab.perm[k]);
    const C zl = gconj(lds_ld(tab.perm[k == 0 ? 0 : L - k]));
    const C e = gscale(gadd(zk, zl), (T)0.5);
    const C dd = gscale(gsub(zk, zl), (T)0.5);
    const C o = gmul(tab.split[k], cmk<T>(dd.y, -dd.x));  // (zk - conj z_{L-k}) / (2i), times exp(-2 pi i k / P)
    T1[(size_t)k * ldT + fr] = gadd(e, o);
    if (2 * k < L) T1[(size_t)(L - k) * ldT + fr] = gconj(gsub(e, o));
  }
}

// ---- pass 2: per frequency column k in [0, P/2]: the n_in stored rows (zero beyond) -> forward
// P-point FFT.  SPEC: store the spectrum column.  Otherwise multiply by the PSF column, inverse
// FFT, store the first n_out rows: T2[k * n_out + i].
//
// The first stage reads the column, the last inverse stage stores it; between them the last forward
// stage, the product and the first inverse stage work on the same r elements and stay in registers.
// The spectrum is stored as they read it: element k of butterfly b at k * (P/r) + b.
template <class T, bool SPEC, int NB>
__global__ __launch_bounds__(kGThreads) void k_g_cols(GColBatch<T, NB> bt, GPlan pl, int n_in, int n_out, int G,
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
  gstage<T, true, false>(pl.r(0), P, P, tab.col, lt, step, column, lds_st);
  int Ls = P / pl.r(0);
  const int last = pl.ns - 1;
  for (int i = 1; i < last; ++i) {
    gstage<T, true, true>(pl.r(i), P, Ls, tab.col, lt, step, lds_ld, lds_st);
    Ls /= pl.r(i);
  }
  C* __restrict__ out = bt.T2[jb] + (size_t)(live ? k : 0) * (SPEC ? P : n_out);
  const C* __restrict__ S = SPEC ? nullptr : bt.S[jb] + (size_t)(live ? k : 0) * P;
  with_radix(pl.r(last), [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    const int nbf = P / R;
    int b = lt;
    C s[R];
    if (!SPEC && b < nbf) {
#pragma unroll
      for (int m = 0; m < R; ++m) s[m] = S[m * nbf + b];
    }
    __syncthreads();
    while (b < nbf) {
      C x[R];
#pragma unroll
      for (int m = 0; m < R; ++m) x[m] = lds_ld(b * R + m);
      GDft<T, R, true>::run(x);
      if (SPEC) {
        if (live) {
#pragma unroll
          for (int m = 0; m < R; ++m) out[m * nbf + b] = x[m];
        }
      } else {
#pragma unroll
        for (int m = 0; m < R; ++m) x[m] = gmul(x[m], s[m]);
        GDft<T, R, false>::run(x);
#pragma unroll
        for (int m = 0; m < R; ++m) lds_st(b * R + m, x[m]);
      }
      b += step;
      if (!SPEC && b < nbf) {
#pragma unroll
        for (int m = 0; m < R; ++m) s[m] = S[m * nbf + b];
      }
    }
  });
  if (SPEC) return;
  for (int i = last - 1; i > 0; --i) {
    Ls *= pl.r(i);
    gstage<T, false, true>(pl.r(i), P, Ls, tab.col, lt, step, lds_ld, lds_st);
  }
  const auto kept = [&](int i, C v) {
    if (live && i < n_out) out[i] = v;
  };
  gstage<T, false, true>(pl.r(0), P, P, tab.col, lt, step, lds_ld, kept);
}

// ---- pass 3: per kept row r: Hermitian half spectrum T2[k * ldT + r], k in [0, P/2] -> the
// P/2-point complex sequence whose inverse FFT interleaves the even and odd output samples, scaled
// by 1/P^2; the first n columns are stored.  Rows share a block as in pass 1; frequencies k and L - k are
// read once for both their elements, and the last stage stores the image.
// VEC: output rows of even length at aligned addresses.
template <class T, bool VEC, int NB>
__global__ __launch_bounds__(kGThreads) void k_g_c2r(GC2rBatch<T, NB> bt, GPlan pl, int n, int ldT, int lg, T scale,
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
  for (int k = lt; 2 * k <= L; k += step) {
    const C xk = T2[(size_t)k * ldT];
    const C xl = gconj(T2[(size_t)(L - k) * ldT]);
    const C s = gadd(xk, xl);
    const C d = gmul(gsub(xk, xl), gconj(tab.split[k]));  // (X_k - conj X_{L-k}) exp(+2 pi i k / P)
    lds_st(tab.perm[k], gadd(s, cmk<T>(-d.y, d.x)));
    if (k > 0 && 2 * k < L) lds_st(tab.perm[L - k], gadd(gconj(s), cmk<T>(d.y, d.x)));
  }
  int Ls = 1;
  for (int i = pl.ns - 1; i > 0; --i) {
    Ls *= pl.r(i);
    gstage<T, false, true>(pl.r(i), L, Ls, tab.row, lt, step, lds_ld, lds_st);
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
  gstage<T, false, true>(pl.r(0), L, L, tab.row, lt, step, lds_ld, image);
}

// ---- host side --------------------------------------------------------------------------------
// The plan of length L: the factors of 2 to 16 with the fewest stages (at least min_stages; each one is a
// pass through LDS and a barrier), of those the one of the smallest sum (the fewest operations).
// Even factors come first and odd ones last: the late stages' LDS strides are multiples of the last radix, and
// odd ones touch all banks.
bool make_gplan(int L, int min_stages, GPlan* p) {
  struct Search {
    int min_stages;
    int cur[kMaxStages], best[kMaxStages];
    int best_n = kMaxStages + 1, best_sum = 0;
    void go(int m, int top, int n, int sum) {
      if (m == 1) {
        if (n >= min_stages && (n < best_n || (n == best_n && sum < best_sum))) {
          best_n = n;
          best_sum = sum;
          std::copy(cur, cur + n, best);
        }
        return;
      }
      if (n == kMaxStages || n >= best_n) return;
      for (int r = std::min(top, m); r >= 2; --r) {
        if (m % r != 0) continue;
        cur[n] = r;
        go(m / r, r, n + 1, sum + r);
      }
    }
  } s;
  s.min_stages = min_stages;
  s.go(L, kMaxRadix, 0, 0);
  if (s.best_n > kMaxStages) return false;
  std::stable_partition(s.best, s.best + s.best_n, [](int r) { return r % 2 == 0; });
  p->L = L;
  p->ns = s.best_n;
  p->code = 0;
  for (int i = 0; i < p->ns; ++i) p->code |= (uint32_t)(s.best[i] - 1) << (4 * i);
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

// stage twiddles of a plan, laid out as gstage reads them, from w[k] = exp(-2 pi i k / P)
template <class C>
void stage_twiddles(const GPlan& pl, const std::vector<C>& w, C* out) {
  const int P = (int)w.size();
  int Ls = pl.L;
  for (int i = 0; i < pl.ns; ++i) {
    const int r = pl.r(i), M = Ls / r, tstep = P / Ls;
    for (int k = 1; k < r; ++k)
      for (int n = 0; n < M; ++n) out[pl.L - Ls + (k - 1) * M + n] = w[(size_t)n * k * tstep];
    Ls = M;
  }
}

// the tables of frame side p in type T (computed in float64), one allocation per device and p
template <class T>
GTables<T> g_tables(int p) {
  using C = Cx<T>;
  const int L = p / 2, n_split = p / 4 + 1;
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
    allow((const void*)k_g_r2c<T, double, false, 1>);
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

template <class T>
void check_g_frame(int p) {
  GPlan pl;
  PMS_REQUIRE(p >= 4 && p % 2 == 0, "FFT frame side must be even and >= 4, got " + std::to_string(p));
  PMS_REQUIRE(p <= gfft_max_frame(sizeof(T)),
              "FFT frame side " + std::to_string(p) + " exceeds the " + std::to_string(gfft_max_frame(sizeof(T))) +
                  " that one LDS transform holds in " + (sizeof(T) == 8 ? "float64" : "float32"));
  PMS_REQUIRE(col_plan(p, &pl) && row_plan(p, &pl),
              "FFT frame side " + std::to_string(p) + " has a prime factor above 13");
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
  GPlan pl;
  return p >= 4 && p % 2 == 0 && p <= gfft_max_frame(real_bytes) && col_plan(p, &pl) && row_plan(p, &pl);
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
