// Direct-stencil IUWT kernels that take two scales a launch, templated on the element type: float32
// planes too small for the row walks (iuwt.hip), and the float64 transforms (iuwt_any.hip).
#pragma once

#include <type_traits>

#include "pms_internal.h"

namespace pms {
namespace {

// Operands of one job of a two-scale recomposition: R_s = h_s (h_{s+1} R + w_{s+1}) + w_s.
template <class T>
struct PairJobT {
  const T* in;           // R_{s+2} (or the coarsest detail plane)
  T* out;                // R_s
  const T* w_in0;        // detail plane of scale s
  const T* w_in1;        // detail plane of scale s+1
  const uint8_t* mask0;  // masks of those planes (null = none)
  const uint8_t* mask1;
  const int* pred;
};
// Operands of one job of a two-scale decomposition: from C_s the detail planes w_s and w_{s+1} and
// the smoothed C_{s+2}; C_{s+1} = h_s C_s exists only in LDS.
template <class T>
struct Dec2JobT {
  const T* in;           // C_s
  T* out_c;              // C_{s+2} (null: not kept)
  T* out_w0;             // w_s
  T* out_w1;             // w_{s+1}
  const uint8_t* mask0;  // masks of w_s and w_{s+1} (null = none)
  const uint8_t* mask1;
  const int* pred;
};

// ---- two scales per launch on small planes ---------------------------------------------------
// Planes in the direct-stencil range take a pair of scales (s, s+1) in one launch.  A workgroup owns
// a tile of one phase class: rows pr + d*i and columns pc + d*j for 16 consecutive lattice indices i
// and j (d = 2^s).  On that lattice scale s is the undilated filter and scale s+1 the same filter at
// spacing 2, so the tile needs its input only within 10 lattice steps (decomposition) or 4
// (recomposition); that region is staged in LDS once, and the intermediate plane -- C_{s+1} of a
// decomposition, T = h_{s+1} R + w_{s+1} of a recomposition -- is computed from it in LDS for the
// tile and a halo of 8 (2) lattice steps and never reaches memory.  Region and halo positions keep
// their unfolded lattice coordinates: a staged input value is the symmetric extension there, and an
// intermediate value at a mirrored position (an odd number of reflections away) accumulates its
// taps in reverse order, which makes it the same sum, in the same order, as the one-scale kernel
// forms at the folded position.  Every plane is therefore bit-identical to two k_iuwt_small launches.
//
// NT threads share a tile (256 or 512, small2_wide): the passes hold 1536 + 1024 + 896 + 512 sums in a
// decomposition and 560 + 400 + 320 + 256 in a recomposition, and each is a chain of dependent LDS reads and
// fmas, so a plane whose tiles do not fill the chip ends sooner with more waves on each.
constexpr int kTile2 = 16;  // tile side in lattice steps

// the B3 filter and its square's taps; both are exact in either type
template <class T>
__device__ __forceinline__ T tap_h5(int k) {
  return k == 2 ? (T)0.375 : (k == 1 || k == 3) ? (T)0.25 : (T)0.0625;
}
template <class T>
__device__ __forceinline__ T tap_h9(int k) {
  constexpr T c[5] = {(T)(1.0 / 256), (T)(8.0 / 256), (T)(28.0 / 256), (T)(56.0 / 256), (T)(70.0 / 256)};
  return c[k < 5 ? k : 8 - k];
}

struct Small2Dims {
  int h, w, d;
  int ntr, ntc;  // tiles per phase along rows and columns
};
template <class J>
struct Small2 {
  template <int NB>
  struct Params : Small2Dims {
    using Dims = Small2Dims;
    J job[NB];  // Dec2Job or PairJob
  };
};

// Folded plane index of lattice coordinates origin + step*(first + k), k in [0, n), for k = lane;
// the index is stored with its mirror flag as ~index when the position lies on a mirrored period.
// Any integer coordinate maps (the extension is periodic with period 2*size).
__device__ __forceinline__ void ext_indices(int* out, int n, int origin, int step, int first, int size) {
  const int k = threadIdx.x & 63;
  if (k < n) {
    const int p = 2 * size;
    int m = (origin + step * (first + k)) % p;
    if (m < 0) m += p;
    out[k] = m >= size ? ~(p - 1 - m) : m;
  }
}
__device__ __forceinline__ int ext_pos(int e) { return e < 0 ? ~e : e; }

// Stage the RS x RS region of lattice positions (ry[i], rx[j]) of plane `in` into LDS rows of RP
// elements.  Every thread issues the same number of loads (the last ones clamped to the final element,
// which is then written twice with the same value), so all of them are in flight together.
template <class T, int RS, int RP, int NT>
__device__ __forceinline__ void stage_region(T* dst, const T* in, const int* ry, const int* rx, int w) {
  constexpr int kPer = (RS * RS + NT - 1) / NT;
  T v[kPer];
  int at[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int e = min((int)threadIdx.x + k * NT, RS * RS - 1);
    const int ri = e / RS, rj = e - ri * RS;
    at[k] = ri * RP + rj;
    v[k] = in[(size_t)ext_pos(ry[ri]) * w + ext_pos(rx[rj])];
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) dst[at[k]] = v[k];
}

// 5-tap sum of v[0], v[step], ... v[4*step] in the order of an unmirrored position, or from v[4*step]
// down to v[0] for a mirrored one: either way the chain adds the taps in the folded position's order.
template <class T>
__device__ __forceinline__ T tap5(const T* v, int step, bool mirrored) {
  T x[5];
#pragma unroll
  for (int b = 0; b < 5; ++b) x[b] = v[b * step];
  T s = 0;
#pragma unroll
  for (int b = 0; b < 5; ++b) s = fma(tap_h5<T>(b), mirrored ? x[4 - b] : x[b], s);
  return s;
}
template <class T>
__device__ __forceinline__ T tap9(const T* v, int step) {
  T s = 0;
#pragma unroll
  for (int b = 0; b < 9; ++b) s = fma(tap_h9<T>(b), v[b * step], s);
  return s;
}

// Scales s and s+1 of a decomposition: w_s, w_{s+1} and (OUTC) C_{s+2} from C_s.  The filters are
// applied separably, row sums first (the one-scale kernel's order): pass 1 forms the 5-tap row sums
// of C_s at every C_{s+1} column and the 9-tap row sums at the tile's columns, pass 2 the column sums
// (C_{s+1} and w_s), pass 3 the row sums of C_{s+1} at spacing 2, pass 4 w_{s+1} and C_{s+2}.
template <class T, bool MASK, bool OUTC, int NB, int NT>
__global__ __launch_bounds__(NT) void k_iuwt_small2_dec(typename Small2<Dec2JobT<T>>::template Params<NB> sp) {
  constexpr int RS = kTile2 + 20, RP = RS + 1;  // staged C_s: lattice -10 .. 25 (rows padded)
  constexpr int IS = kTile2 + 16, IP = IS + 1;  // C_{s+1}: lattice -8 .. 23
  constexpr int N5 = RS * IS;                   // pass 1: 5-tap row sums, every staged row
  constexpr int N9 = (kTile2 + 8) * kTile2;     // pass 1: 9-tap row sums, staged rows 6 .. 29
  constexpr int M9 = IS * kTile2;               // pass 3: 9-tap row sums of C_{s+1}, every row
  constexpr int M5 = (kTile2 + 8) * kTile2;     // pass 3: 5-tap row sums of C_{s+1}, rows 4 .. 27
  constexpr int TT = kTile2 * kTile2;
  static_assert(N5 % 64 == 0 && N9 % 64 == 0 && M9 % 64 == 0 && NT % TT == 0, "passes split wave-uniformly");
  static_assert(IS * IS % NT == 0, "pass 2 splits evenly");
  static_assert(M9 + M5 <= RS * IP, "pass 3 reuses the pass-1 array");
  __shared__ T cs[RS * RP];
  __shared__ T hs[RS * IP];  // pass 1 5-tap sums [row][column]; pass 3 sums afterwards
  __shared__ T h9[N9];
  __shared__ T c1[IS * IP];
  __shared__ int ry[RS], rx[RS];
  const Dec2JobT<T> a = sp.job[blockIdx.z];
  if (a.pred && *a.pred == 0) return;
  const int h = sp.h, w = sp.w, d = sp.d;
  const int pr = blockIdx.y / sp.ntr, i0 = (blockIdx.y - pr * sp.ntr) * kTile2;
  const int pc = blockIdx.x / sp.ntc, j0 = (blockIdx.x - pc * sp.ntc) * kTile2;
  if (threadIdx.x < 64)
    ext_indices(ry, RS, pr, d, i0 - 10, h);
  else if (threadIdx.x < 128)
    ext_indices(rx, RS, pc, d, j0 - 10, w);
  // this thread's pixel: with 256 threads every output, with more w_{s+1} (and w_s) in the first 256 threads
  // and C_{s+2} in the next
  const int part = threadIdx.x / TT, px = threadIdx.x % TT;
  const int ty = px / kTile2, tx = px % kTile2;
  const int row = pr + d * (i0 + ty), col = pc + d * (j0 + tx);
  const bool live = row < h && col < w && part < 2;
  const size_t off = live ? (size_t)row * w + col : 0;
  const bool keep0 = !MASK || part > 0 || a.mask0[off] != 0;
  const bool keep1 = !MASK || part > 0 || a.mask1[off] != 0;
  __syncthreads();
  stage_region<T, RS, RP, NT>(cs, a.in, ry, rx, w);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < (N5 + N9 + NT - 1) / NT; ++k) {
    const int e = threadIdx.x + k * NT;
    if (e < N5) {
      const int ri = e / IS, v = e - ri * IS;
      hs[ri * IP + v] = tap5(cs + ri * RP + v, 1, rx[v + 2] < 0);
    } else if (e < N5 + N9) {
      const int f = e - N5, ri = f / kTile2, x = f - ri * kTile2;
      h9[f] = tap9(cs + (ri + 6) * RP + x + 6, 1);
    }
  }
  __syncthreads();
  // C_{s+1} slot (u, v) is centred on staged (u + 2, v + 2); w_s on staged (ty + 10, tx + 10)
#pragma unroll
  for (int k = 0; k < IS * IS / NT; ++k) {
    const int e = threadIdx.x + k * NT;
    const int u = e / IS, v = e - u * IS;
    c1[u * IP + v] = tap5(hs + u * IP + v, IP, ry[u + 2] < 0);
  }
  if (live && part == 0)
    a.out_w0[off] = keep0 ? cs[(ty + 10) * RP + tx + 10] - tap9(h9 + ty * kTile2 + tx, kTile2) : (T)0;
  __syncthreads();
  T* g9 = hs;       // [32][16]: 9-tap sums at spacing 2 of C_{s+1} row r at tile column x
  T* g5 = hs + M9;  // [24][16]: 5-tap sums of C_{s+1} row r + 4
#pragma unroll
  for (int k = 0; k < (M9 + M5 + NT - 1) / NT; ++k) {
    const int e = threadIdx.x + k * NT;
    if (e < M9) {
      const int r = e / kTile2, x = e - r * kTile2;
      g9[e] = tap9(c1 + r * IP + x, 2);
    } else if (OUTC && e < M9 + M5) {
      const int f = e - M9, r = f / kTile2, x = f - r * kTile2;
      g5[f] = tap5(c1 + (r + 4) * IP + x + 4, 2, false);
    }
  }
  __syncthreads();
  if (!live) return;
  // w_{s+1} centred on slot (ty + 8, tx + 8), taps on slot rows ty + 2i; C_{s+2} on rows ty + 4 + 2k
  if (part == 0)
    a.out_w1[off] = keep1 ? c1[(ty + 8) * IP + tx + 8] - tap9(g9 + ty * kTile2 + tx, 2 * kTile2) : (T)0;
  if (OUTC && (NT == TT || part == 1)) a.out_c[off] = tap5(g5 + ty * kTile2 + tx, 2 * kTile2, false);
}

// Scales s+1 then s of a recomposition: R_s = h_s T + w_s with T = h_{s+1} R + w_{s+1}.  Pass 1 forms
// the row sums of R at spacing 2 at every T column, pass 2 T, pass 3 the row sums of T at the tile's
// columns, pass 4 R_s.
template <class T, bool MASK, int NB, int NT>
__global__ __launch_bounds__(NT) void k_iuwt_small2_rec(typename Small2<PairJobT<T>>::template Params<NB> sp) {
  constexpr int RS = kTile2 + 12, RP = RS + 1;  // staged R: lattice -6 .. 21
  constexpr int TS = kTile2 + 4, TP = TS + 1;   // T: lattice -2 .. 17
  constexpr int N1 = RS * TS;                   // pass 1 sums
  constexpr int N2 = TS * TS;                   // T slots
  constexpr int N3 = TS * kTile2;               // pass 3 sums
  constexpr int K2 = (N2 + NT - 1) / NT;
  constexpr int TT = kTile2 * kTile2;
  __shared__ T rs[RS * RP];
  __shared__ T hr[RS * TP];  // pass 1 sums [row][T column]; pass 3 sums afterwards
  __shared__ T tt[TS * TP];
  __shared__ int ry[RS], rx[RS];
  const PairJobT<T> a = sp.job[blockIdx.z];
  if (a.pred && *a.pred == 0) return;
  const int h = sp.h, w = sp.w, d = sp.d;
  const int pr = blockIdx.y / sp.ntr, i0 = (blockIdx.y - pr * sp.ntr) * kTile2;
  const int pc = blockIdx.x / sp.ntc, j0 = (blockIdx.x - pc * sp.ntc) * kTile2;
  if (threadIdx.x < 64)
    ext_indices(ry, RS, pr, d, i0 - 6, h);
  else if (threadIdx.x < 128)
    ext_indices(rx, RS, pc, d, j0 - 6, w);
  const int ty = threadIdx.x / kTile2, tx = threadIdx.x % kTile2;
  const int row = pr + d * (i0 + ty), col = pc + d * (j0 + tx);
  const bool live = threadIdx.x < TT && row < h && col < w;
  const size_t off = live ? (size_t)row * w + col : 0;
  T wi0 = a.w_in0[off];
  if (MASK && a.mask0[off] == 0) wi0 = 0;
  __syncthreads();
  // the detail term of T slot (u, v) (staged (u + 4, v + 4)) is read at the folded position, where
  // the one-scale launch adds it; the last slots are clamped (a repeated slot writes the same value)
  T wi1[K2];
#pragma unroll
  for (int k = 0; k < K2; ++k) {
    const int e = min((int)threadIdx.x + k * NT, N2 - 1);
    const int u = e / TS, v = e - u * TS;
    const size_t o = (size_t)ext_pos(ry[u + 4]) * w + ext_pos(rx[v + 4]);
    wi1[k] = a.w_in1[o];
    if (MASK && a.mask1[o] == 0) wi1[k] = 0;
  }
  stage_region<T, RS, RP, NT>(rs, a.in, ry, rx, w);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < (N1 + NT - 1) / NT; ++k) {
    const int e = min((int)threadIdx.x + k * NT, N1 - 1);
    const int ri = e / TS, v = e - ri * TS;
    hr[ri * TP + v] = tap5(rs + ri * RP + v, 2, rx[v + 4] < 0);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K2; ++k) {
    const int e = min((int)threadIdx.x + k * NT, N2 - 1);
    const int u = e / TS, v = e - u * TS;
    tt[u * TP + v] = tap5(hr + u * TP + v, 2 * TP, ry[u + 4] < 0) + wi1[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < (N3 + NT - 1) / NT; ++k) {
    const int e = min((int)threadIdx.x + k * NT, N3 - 1);
    const int r = e / kTile2, x = e - r * kTile2;
    hr[e] = tap5(tt + r * TP + x, 1, false);
  }
  __syncthreads();
  if (!live) return;
  a.out[off] = tap5(hr + ty * kTile2 + tx, kTile2, false) + wi0;
}

template <class J>
using Small2Batch = typename Small2<J>::template Params<kMaxBatch>;

template <class J>
Small2Batch<J> small2_params(int h, int w, int s) {
  Small2Batch<J> sp{};
  sp.h = h;
  sp.w = w;
  sp.d = 1 << s;
  sp.ntr = ceil_div(ceil_div(h, sp.d), kTile2);
  sp.ntc = ceil_div(ceil_div(w, sp.d), kTile2);
  return sp;
}

dim3 small2_grid(const Small2Dims& sp, int nb) { return dim3(sp.d * sp.ntc, sp.d * sp.ntr, nb); }

// Threads per tile: 512 while a launch has at most two tiles per CU, whose latency is then its time; 256 beyond,
// where the chip is full either way.  A pair of float32 decomposition scales of a 256^2 plane (256 tiles)
// takes 4.5 us with 512 and 5.4 with 256 threads (1024: 4.5), a recomposition 3.7 and 3.9; a float64 pair of a
// 512^2 plane (1024 tiles) 9.1 and 9.2, 6.4 and 5.9; a batch of sixteen 256^2 planes 18.7 and 16.3.
inline bool small2_wide(dim3 g) { return (long)g.x * g.y * g.z <= 512; }

// jobs[0..count) share shape and scale pair; masked and unmasked jobs, and jobs that keep C_{s+2}
// and those that do not, go to separate launches
template <class T>
void small2_dec_batch(const Dec2JobT<T>* jobs, int count, int h, int w, int s, hipStream_t st) {
  Small2Batch<Dec2JobT<T>> sp = small2_params<Dec2JobT<T>>(h, w, s);
  for (int kind = 0; kind < 4; ++kind) {
    const bool masked = (kind & 1) != 0, keep_c = (kind & 2) != 0;
    int nb = 0;
    auto flush = [&]() {
      if (nb == 0) return;
      const dim3 g = small2_grid(sp, nb);
      with_jobs<Small2<Dec2JobT<T>>::template Params>(sp, nb, [&](const auto& p) {
        constexpr int NB = sizeof(p.job) / sizeof(p.job[0]);
        auto go = [&](auto nt) {
          constexpr int NT = decltype(nt)::value;
          switch (kind) {
            case 0: hipLaunchKernelGGL((k_iuwt_small2_dec<T, false, false, NB, NT>), g, dim3(NT), 0, st, p); break;
            case 1: hipLaunchKernelGGL((k_iuwt_small2_dec<T, true, false, NB, NT>), g, dim3(NT), 0, st, p); break;
            case 2: hipLaunchKernelGGL((k_iuwt_small2_dec<T, false, true, NB, NT>), g, dim3(NT), 0, st, p); break;
            default: hipLaunchKernelGGL((k_iuwt_small2_dec<T, true, true, NB, NT>), g, dim3(NT), 0, st, p); break;
          }
        };
        small2_wide(g) ? go(std::integral_constant<int, 512>{}) : go(std::integral_constant<int, 256>{});
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
void small2_rec_batch(const PairJobT<T>* jobs, int count, int h, int w, int s, hipStream_t st) {
  Small2Batch<PairJobT<T>> sp = small2_params<PairJobT<T>>(h, w, s);
  for (int masked = 0; masked < 2; ++masked) {
    int nb = 0;
    auto flush = [&]() {
      if (nb == 0) return;
      const dim3 g = small2_grid(sp, nb);
      with_jobs<Small2<PairJobT<T>>::template Params>(sp, nb, [&](const auto& p) {
        constexpr int NB = sizeof(p.job) / sizeof(p.job[0]);
        auto go = [&](auto nt) {
          constexpr int NT = decltype(nt)::value;
          if (masked)
            hipLaunchKernelGGL((k_iuwt_small2_rec<T, true, NB, NT>), g, dim3(NT), 0, st, p);
          else
            hipLaunchKernelGGL((k_iuwt_small2_rec<T, false, NB, NT>), g, dim3(NT), 0, st, p);
        };
        small2_wide(g) ? go(std::integral_constant<int, 512>{}) : go(std::integral_constant<int, 256>{});
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

}  // namespace
}  // namespace pms
