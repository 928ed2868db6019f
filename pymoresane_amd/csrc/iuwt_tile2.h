// Two IUWT scales a launch on tiles of 32 x 32 lattice positions: the form of iuwt_small2.h's kernels for
// float32 launches that fill the chip (in float64 its LDS holds half the blocks, and it measured no faster).
//
// The lattice, the staged region, the intermediate plane in LDS and the order of every sum are those of
// iuwt_small2.h (so the planes are the same bits); what differs is the work per output.  The 16 x 16 tile reads
// 5.1 (decomposition) or 3.1 (recomposition) inputs and forms 15.5 or 6 sums per output, each from its own LDS
// reads: about 105 reads an output.  The 32 x 32 tile takes 2.6 or 1.9 inputs and 10.7 or 4.9 sums, and a
// thread forms 4 to 8 neighbouring sums from one window of the row or column in registers: about 20
// reads.  Sums of a mirrored position add their taps from the other end; only tiles that touch a border
// hold any, so the others run without the test.  Tiles of one place and all phases are neighbours on one XCD:
// their inputs share cache lines, and their partial-line stores meet in one L2.  C_{s+1} takes the place of the staged
// region: 26 KB a block, six blocks a CU (with 36 KB and four the pair (0,1) of a 4096^2 plane took 131 us, with 26 KB 89 us).
// At that size vector instructions (4.0e7 waves' worth, 65 us at one a cycle and SIMD group) and LDS accesses (45 us)
// bound it; the row walks take 86 us there and keep the larger planes.
#pragma once

#include "iuwt_small2.h"

namespace pms {

bool tile2_fits(int h, int w, int s, int jobs, bool recomp);  // iuwt.hip

namespace {

constexpr int kTile32 = 32;
constexpr int kTileThreads = 320;

template <class J>
struct Tile2 {
  template <int NB>
  struct Params : Small2Dims {
    using Dims = Small2Dims;
    J job[NB];
  };
};

struct TilePos {
  int pr, i0, pc, j0;
};
// block -> tile: places along a row of tiles, then down, all d x d phases of a place side by side
__device__ __forceinline__ TilePos tile_pos(const Small2Dims& sp) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const unsigned dd = (unsigned)(sp.d * sp.d);
  const unsigned place = b / dd, phase = b - place * dd;
  const unsigned tr = place / (unsigned)sp.ntc, tc = place - tr * (unsigned)sp.ntc;
  const unsigned pr = phase / (unsigned)sp.d, pc = phase - pr * (unsigned)sp.d;
  return {(int)pr, (int)tr * kTile32, (int)pc, (int)tc * kTile32};
}
// whether the lattice positions first .. first + n - 1 from origin leave [0, size)
__device__ __forceinline__ bool tile_leaves(int origin, int d, int first, int n, int size) {
  return origin + d * first < 0 || origin + d * (first + n - 1) >= size;
}

// The tile's outputs: plane element (row, column) = origin + lane part, the first in a scalar register, the second a
// 32-bit byte offset (planes have at most 2^29 elements), and the lattice rows and columns that exist.
struct TileOut {
  size_t origin;       // element of lattice (i0, j0)
  unsigned pitch;      // elements from one lattice row to the next
  int rows, cols;      // lattice rows and columns from (i0, j0) on
};
__device__ __forceinline__ TileOut tile_out(const Small2Dims& sp, const TilePos& tp) {
  TileOut o;
  o.origin = (size_t)(tp.pr + sp.d * tp.i0) * sp.w + (tp.pc + sp.d * tp.j0);
  o.pitch = (unsigned)sp.d * (unsigned)sp.w;
  o.rows = (sp.h - tp.pr + sp.d - 1) / sp.d - tp.i0;
  o.cols = (sp.w - tp.pc + sp.d - 1) / sp.d - tp.j0;
  return o;
}
// element k lattice rows below the lane's own (its offset from the tile's origin is `lane`)
template <class T>
__device__ __forceinline__ T* tile_at(T* plane, const TileOut& o, unsigned lane, int k) {
  return reinterpret_cast<T*>(reinterpret_cast<char*>(const_cast<std::remove_const_t<T>*>(plane) + o.origin + (size_t)k * o.pitch) +
                              lane * (unsigned)sizeof(T));
}

// Stage the RS x RS region of lattice positions (ry[i], rx[j]) of plane `in` into LDS rows of RP elements: a wave
// takes whole rows, so a row's address is scalar and a lane's column is read once.  Every thread issues the same
// number of loads (the last ones clamped to the final row or column, which is then written twice with the same value).
template <class T, int RS, int RP, int NT>
__device__ __forceinline__ void stage_rows(T* dst, const T* __restrict__ in, const int* ry, const int* rx, int w) {
  constexpr int NW = NT / 64, kPer = (RS + NW - 1) / NW;
  const int c = min((int)(threadIdx.x & 63), RS - 1);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const unsigned col = (unsigned)ext_pos(rx[c]);
  T v[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int row = __builtin_amdgcn_readfirstlane(ext_pos(ry[min(wave + k * NW, RS - 1)]));
    v[k] = (in + (size_t)row * w)[col];
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) dst[min(wave + k * NW, RS - 1) * RP + c] = v[k];
}

// N values from an LDS address that is a multiple of G values (G * sizeof(T) bytes <= 16)
template <class T, int N, int G>
__device__ __forceinline__ void lds_window(T (&x)[N], const T* p) {
  struct alignas(G * sizeof(T)) V {
    T a[G];
  };
  static_assert(N % G == 0, "whole vectors");
#pragma unroll
  for (int k = 0; k < N / G; ++k) {
    const V v = reinterpret_cast<const V*>(p)[k];
#pragma unroll
    for (int i = 0; i < G; ++i) x[k * G + i] = v.a[i];
  }
}
template <class T, int N, int G>
__device__ __forceinline__ void lds_put(T* p, const T (&x)[N]) {
  struct alignas(G * sizeof(T)) V {
    T a[G];
  };
#pragma unroll
  for (int k = 0; k < N / G; ++k) {
    V v;
#pragma unroll
    for (int i = 0; i < G; ++i) v.a[i] = x[k * G + i];
    reinterpret_cast<V*>(p)[k] = v;
  }
}
template <class T>
constexpr int lds_wide() {
  return 16 / (int)sizeof(T);
}

// 5- and 9-tap sums of x[at], x[at + step], ... in iuwt_small2.h's order
template <int step, class T, int N>
__device__ __forceinline__ T win5(const T (&x)[N], int at, bool mirrored) {
  T s = 0;
#pragma unroll
  for (int b = 0; b < 5; ++b) s = fma(tap_h5<T>(b), mirrored ? x[at + step * (4 - b)] : x[at + step * b], s);
  return s;
}
template <int step, class T, int N>
__device__ __forceinline__ T win9(const T (&x)[N], int at) {
  T s = 0;
#pragma unroll
  for (int b = 0; b < 9; ++b) s = fma(tap_h9<T>(b), x[at + step * b], s);
  return s;
}

// Scales s and s+1 of a decomposition.  Pass 1: row sums of C_s, 5 taps at the 48 columns of C_{s+1} and 9
// taps at the tile's; pass 2: column sums, C_{s+1} and w_s; pass 3: row sums of C_{s+1} at spacing 2;
// pass 4: w_{s+1} and C_{s+2}.
template <class T, bool MASK, bool OUTC, int NB>
__global__ __launch_bounds__(kTileThreads) void k_iuwt_tile2_dec(typename Tile2<Dec2JobT<T>>::template Params<NB> sp) {
  constexpr int TS = kTile32;
  constexpr int RS = TS + 20, RP = RS;  // staged C_s: lattice -10 .. 41
  constexpr int IS = TS + 16, IP = IS;  // C_{s+1}: lattice -8 .. 39
  constexpr int R9 = TS + 8;            // rows of 9-tap sums: staged 6 .. 45
  constexpr int W = lds_wide<T>() > 4 ? 4 : lds_wide<T>();
  static_assert(IS * TS + R9 * TS <= RS * IP + R9 * TS, "pass 3 reuses the pass-1 arrays");
  __shared__ __attribute__((aligned(16))) T cs[RS * RP];            // C_s; C_{s+1} after pass 1
  __shared__ __attribute__((aligned(16))) T hs[RS * IP + R9 * TS];  // pass 1 sums; pass 3 sums afterwards
  static_assert(IS * IP <= RS * RP, "C_{s+1} fits where C_s was");
  T* c1 = cs;
  __shared__ int ry[RS], rx[RS];
  T* h9 = hs + RS * IP;
  const Dec2JobT<T> a = sp.job[blockIdx.y];
  if (a.pred && *a.pred == 0) return;
  const int h = sp.h, w = sp.w, d = sp.d;
  const TilePos tp = tile_pos(sp);
  const int tid = threadIdx.x;
  if (tid < 64)
    ext_indices(ry, RS, tp.pr, d, tp.i0 - 10, h);
  else if (tid < 128)
    ext_indices(rx, RS, tp.pc, d, tp.j0 - 10, w);
  // outputs of threads 0 .. 255: column ox; rows 4 og .. + 3 of w_s, rows 8 (og / 2) + og % 2 + {0, 2, 4, 6} of
  // w_{s+1} and C_{s+2}
  const int ox = tid & (TS - 1), og = tid / TS;
  const int y0 = 4 * og, y1 = 8 * (og >> 1) + (og & 1);
  const TileOut to = tile_out(sp, tp);
  const bool owner = tid < TS * 8 && ox < to.cols;
  const unsigned at0 = (unsigned)y0 * to.pitch + (unsigned)(d * ox), at1 = (unsigned)y1 * to.pitch + (unsigned)(d * ox);
  bool keep0[4], keep1[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    keep0[k] = keep1[k] = true;
    if (MASK) {
      if (owner && y0 + k < to.rows) keep0[k] = *tile_at(a.mask0, to, at0, k) != 0;
      if (owner && y1 + 2 * k < to.rows) keep1[k] = *tile_at(a.mask1, to, at1, 2 * k) != 0;
    }
  }
  __syncthreads();
  stage_rows<T, RS, RP, kTileThreads>(cs, a.in, ry, rx, w);
  __syncthreads();
  T centre[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) centre[k] = tid < TS * 8 ? cs[(y0 + k + 10) * RP + ox + 10] : (T)0;
  const bool border = tile_leaves(tp.pr, d, tp.i0 - 10, RS, h) || tile_leaves(tp.pc, d, tp.j0 - 10, RS, w);
  const auto passes12 = [&](auto bc) {
    constexpr bool B = decltype(bc)::value;
    // 4 columns of the 5-tap sums from 8 staged ones; 4 of the 9-tap sums from 12
    for (int e = tid; e < RS * (IS / 4); e += kTileThreads) {
      const int r = e / (IS / 4), q = e - r * (IS / 4);
      T x[8], s[4];
      lds_window<T, 8, W>(x, cs + r * RP + 4 * q);
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] = win5<1>(x, i, B && rx[4 * q + i + 2] < 0);
      lds_put<T, 4, W>(hs + r * IP + 4 * q, s);
    }
    for (int e = tid; e < R9 * (TS / 4); e += kTileThreads) {
      const int r = e / (TS / 4), q = e - r * (TS / 4);
      T x[12], s[4];
      lds_window<T, 12, 2>(x, cs + (r + 6) * RP + 4 * q + 6);
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] = win9<1>(x, i);
      lds_put<T, 4, W>(h9 + r * TS + 4 * q, s);
    }
    __syncthreads();
    // 8 rows of a column of C_{s+1} from 12 row sums
    for (int e = tid; e < (IS / 8) * IS; e += kTileThreads) {
      const int g = e / IS, v = e - g * IS;
      T x[12];
#pragma unroll
      for (int i = 0; i < 12; ++i) x[i] = hs[(8 * g + i) * IP + v];
#pragma unroll
      for (int i = 0; i < 8; ++i) c1[(8 * g + i) * IP + v] = win5<1>(x, i, B && ry[8 * g + i + 2] < 0);
    }
  };
  if (border)
    passes12(std::true_type{});
  else
    passes12(std::false_type{});
  if (owner) {
    T x[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) x[i] = h9[(y0 + i) * TS + ox];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const T v = centre[k] - win9<1>(x, k);
      if (y0 + k < to.rows) *tile_at(a.out_w0, to, at0, k) = keep0[k] ? v : (T)0;
    }
  }
  __syncthreads();
  T* g9 = hs;            // [48][32]: 9-tap sums at spacing 2 of C_{s+1}
  T* g5 = hs + IS * TS;  // [40][32]: 5-tap sums of C_{s+1} row r + 4
  for (int e = tid; e < IS * (TS / 8); e += kTileThreads) {
    const int r = e / (TS / 8), q = e - r * (TS / 8);
    T x[24], s[8];
    lds_window<T, 24, W>(x, c1 + r * IP + 8 * q);
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = win9<2>(x, i);
    lds_put<T, 8, W>(g9 + r * TS + 8 * q, s);
    if (OUTC && r >= 4 && r < 4 + R9) {
#pragma unroll
      for (int i = 0; i < 8; ++i) s[i] = win5<2>(x, i + 4, false);
      lds_put<T, 8, W>(g5 + (r - 4) * TS + 8 * q, s);
    }
  }
  __syncthreads();
  if (!owner) return;
  {
    T x[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) x[i] = g9[(y1 + 2 * i) * TS + ox];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const T v = c1[(y1 + 2 * k + 8) * IP + ox + 8] - win9<1>(x, k);
      if (y1 + 2 * k < to.rows) *tile_at(a.out_w1, to, at1, 2 * k) = keep1[k] ? v : (T)0;
    }
  }
  if (OUTC) {
    T x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = g5[(y1 + 2 * i) * TS + ox];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (y1 + 2 * k < to.rows) *tile_at(a.out_c, to, at1, 2 * k) = win5<1>(x, k, false);
  }
}

// Scales s+1 then s of a recomposition.  Pass 1: row sums of R at spacing 2 at the 36 columns of T; pass 2: T;
// pass 3: row sums of T at the tile's columns; pass 4: R_s.
template <class T, bool MASK, int NB>
__global__ __launch_bounds__(kTileThreads) void k_iuwt_tile2_rec(typename Tile2<PairJobT<T>>::template Params<NB> sp) {
  constexpr int TS = kTile32;
  constexpr int RS = TS + 12, RP = RS;  // staged R: lattice -6 .. 37
  constexpr int US = TS + 4, UP = US;   // T: lattice -2 .. 33
  constexpr int W = lds_wide<T>() > 4 ? 4 : lds_wide<T>();
  __shared__ __attribute__((aligned(16))) T rs[RS * RP];
  __shared__ __attribute__((aligned(16))) T hr[RS * UP];  // pass 1 sums [row][T column]; pass 3 sums afterwards
  __shared__ __attribute__((aligned(16))) T tt[US * US];
  __shared__ int ry[RS], rx[RS];
  const PairJobT<T> a = sp.job[blockIdx.y];
  if (a.pred && *a.pred == 0) return;
  const int h = sp.h, w = sp.w, d = sp.d;
  const TilePos tp = tile_pos(sp);
  const int tid = threadIdx.x;
  if (tid < 64)
    ext_indices(ry, RS, tp.pr, d, tp.i0 - 6, h);
  else if (tid < 128)
    ext_indices(rx, RS, tp.pc, d, tp.j0 - 6, w);
  const int ox = tid & (TS - 1), y0 = 4 * (tid / TS);
  const TileOut to = tile_out(sp, tp);
  const bool owner = tid < TS * 8 && ox < to.cols;
  const unsigned at0 = (unsigned)y0 * to.pitch + (unsigned)(d * ox);
  T wi0[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    wi0[k] = 0;
    if (owner && y0 + k < to.rows) {
      wi0[k] = *tile_at(a.w_in0, to, at0, k);
      if (MASK && *tile_at(a.mask0, to, at0, k) == 0) wi0[k] = 0;
    }
  }
  __syncthreads();
  // T slots of threads 0 .. 215: column tv, rows tu + {0, 2, 4, 6, 8, 10}, the detail term read at the folded position
  const int tg = tid / US, tv = tid - tg * US;
  const bool slots = tid < 6 * US;
  const int tu = 12 * (tg >> 1) + (tg & 1);
  T wi1[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const int u = slots ? tu + 2 * k : 0, v = slots ? tv : 0;
    const size_t o = (size_t)ext_pos(ry[u + 4]) * w + ext_pos(rx[v + 4]);
    wi1[k] = a.w_in1[o];
    if (MASK && a.mask1[o] == 0) wi1[k] = 0;
  }
  stage_rows<T, RS, RP, kTileThreads>(rs, a.in, ry, rx, w);
  __syncthreads();
  const bool border = tile_leaves(tp.pr, d, tp.i0 - 6, RS, h) || tile_leaves(tp.pc, d, tp.j0 - 6, RS, w);
  const auto passes12 = [&](auto bc) {
    constexpr bool B = decltype(bc)::value;
    // 4 columns of the row sums from 12 staged ones
    for (int e = tid; e < RS * (US / 4); e += kTileThreads) {
      const int r = e / (US / 4), q = e - r * (US / 4);
      T x[12], s[4];
      lds_window<T, 12, W>(x, rs + r * RP + 4 * q);
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] = win5<2>(x, i, B && rx[4 * q + i + 4] < 0);
      lds_put<T, 4, W>(hr + r * UP + 4 * q, s);
    }
    __syncthreads();
    if (slots) {
      T x[10];
#pragma unroll
      for (int i = 0; i < 10; ++i) x[i] = hr[(tu + 2 * i) * UP + tv];
#pragma unroll
      for (int k = 0; k < 6; ++k) tt[(tu + 2 * k) * US + tv] = win5<1>(x, k, B && ry[tu + 2 * k + 4] < 0) + wi1[k];
    }
  };
  if (border)
    passes12(std::true_type{});
  else
    passes12(std::false_type{});
  __syncthreads();
  for (int e = tid; e < US * (TS / 4); e += kTileThreads) {
    const int r = e / (TS / 4), q = e - r * (TS / 4);
    T x[8], s[4];
    lds_window<T, 8, W>(x, tt + r * US + 4 * q);
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = win5<1>(x, i, false);
    lds_put<T, 4, W>(hr + r * TS + 4 * q, s);
  }
  __syncthreads();
  if (!owner) return;
  T x[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = hr[(y0 + i) * TS + ox];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (y0 + k < to.rows) *tile_at(a.out, to, at0, k) = win5<1>(x, k, false) + wi0[k];
}

template <class J>
using Tile2Batch = typename Tile2<J>::template Params<kMaxBatch>;

template <class J>
Tile2Batch<J> tile2_params(int h, int w, int s) {
  Tile2Batch<J> sp{};
  sp.h = h;
  sp.w = w;
  sp.d = 1 << s;
  sp.ntr = ceil_div(ceil_div(h, sp.d), kTile32);
  sp.ntc = ceil_div(ceil_div(w, sp.d), kTile32);
  return sp;
}
// 32 x 32 tiles of one plane at scales (s, s+1)
inline long tile2_tiles(int h, int w, int s) {
  const long d = 1L << s;
  return d * d * ceil_div(ceil_div(h, (int)d), kTile32) * ceil_div(ceil_div(w, (int)d), kTile32);
}

// jobs[0..count) share shape and scale pair, as in iuwt_small2.h
template <class T>
void tile2_dec_batch(const Dec2JobT<T>* jobs, int count, int h, int w, int s, hipStream_t st) {
  Tile2Batch<Dec2JobT<T>> sp = tile2_params<Dec2JobT<T>>(h, w, s);
  const unsigned tiles = (unsigned)tile2_tiles(h, w, s);
  for (int kind = 0; kind < 4; ++kind) {
    const bool masked = (kind & 1) != 0, keep_c = (kind & 2) != 0;
    int nb = 0;
    auto flush = [&]() {
      if (nb == 0) return;
      const dim3 g(tiles, nb), b(kTileThreads);
      with_jobs<Tile2<Dec2JobT<T>>::template Params>(sp, nb, [&](const auto& p) {
        constexpr int NB = sizeof(p.job) / sizeof(p.job[0]);
        switch (kind) {
          case 0: hipLaunchKernelGGL((k_iuwt_tile2_dec<T, false, false, NB>), g, b, 0, st, p); break;
          case 1: hipLaunchKernelGGL((k_iuwt_tile2_dec<T, true, false, NB>), g, b, 0, st, p); break;
          case 2: hipLaunchKernelGGL((k_iuwt_tile2_dec<T, false, true, NB>), g, b, 0, st, p); break;
          default: hipLaunchKernelGGL((k_iuwt_tile2_dec<T, true, true, NB>), g, b, 0, st, p); break;
        }
      });
      PMS_LAUNCH_CHECK();
      nb = 0;
    };
    for (int k = 0; k < count; ++k) {
      if ((jobs[k].mask0 != nullptr) != masked || (jobs[k].out_c != nullptr) != keep_c) continue;
      PMS_REQUIRE(jobs[k].out_w0 && jobs[k].out_w1 && (!masked || jobs[k].mask1),
                  "two-scale decomposition needs both detail planes (and both masks or none)");
      sp.job[nb++] = jobs[k];
      if (nb == kMaxBatch) flush();
    }
    flush();
  }
}

template <class T>
void tile2_rec_batch(const PairJobT<T>* jobs, int count, int h, int w, int s, hipStream_t st) {
  Tile2Batch<PairJobT<T>> sp = tile2_params<PairJobT<T>>(h, w, s);
  const unsigned tiles = (unsigned)tile2_tiles(h, w, s);
  for (int masked = 0; masked < 2; ++masked) {
    int nb = 0;
    auto flush = [&]() {
      if (nb == 0) return;
      const dim3 g(tiles, nb), b(kTileThreads);
      with_jobs<Tile2<PairJobT<T>>::template Params>(sp, nb, [&](const auto& p) {
        constexpr int NB = sizeof(p.job) / sizeof(p.job[0]);
        if (masked)
          hipLaunchKernelGGL((k_iuwt_tile2_rec<T, true, NB>), g, b, 0, st, p);
        else
          hipLaunchKernelGGL((k_iuwt_tile2_rec<T, false, NB>), g, b, 0, st, p);
      });
      PMS_LAUNCH_CHECK();
      nb = 0;
    };
    for (int k = 0; k < count; ++k) {
      if ((jobs[k].mask0 != nullptr) != (masked != 0)) continue;
      PMS_REQUIRE(!masked || jobs[k].mask1, "two-scale recomposition needs both masks or none");
      sp.job[nb++] = jobs[k];
      if (nb == kMaxBatch) flush();
    }
    flush();
  }
}

// a pair's launch with the tile size that tile2_fits names (32 or 16)
template <class T>
void pair_dec_batch(const Dec2JobT<T>* jobs, int count, int h, int w, int s, hipStream_t st) {
  if (tile2_fits(h, w, s, count, false))
    tile2_dec_batch<T>(jobs, count, h, w, s, st);
  else
    small2_dec_batch<T>(jobs, count, h, w, s, st);
}
template <class T>
void pair_rec_batch(const PairJobT<T>* jobs, int count, int h, int w, int s, hipStream_t st) {
  if (tile2_fits(h, w, s, count, true))
    tile2_rec_batch<T>(jobs, count, h, w, s, st);
  else
    small2_rec_batch<T>(jobs, count, h, w, s, st);
}

}  // namespace
}  // namespace pms
