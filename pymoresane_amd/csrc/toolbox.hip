// Noise estimate, thresholding, source extraction and the vector/scalar
// kernels of the conjugate-gradient minor loop, for gfx950.
//
// Semantics follow pymoresane/iuwt_toolbox.py:
//   estimate_threshold (17-48) : median(|w| over the noise mask) / 0.6745,
//                                exact: selection by the float bits of |w|
//                                (non-negative floats order like unsigned ints),
//                                in one reading of the planes through a sampled
//                                range of keys, or as a radix select where there
//                                is no workspace for that; np.median's mean of
//                                the two middle values for even counts;
//   apply_threshold (50-75)    : w where |w| > sigma * t (strict), else 0;
//   source_extraction (97-154) : 8-connected labels of non-zero pixels by
//                                union-find with atomicMin links (every root is
//                                its component's smallest raster index, so the
//                                partition and the raster-order label numbering
//                                are exactly scipy.ndimage.label's), then the
//                                coarse-to-fine keep rule on the device;
//   snr_ratio (292-306)        : float64 sums of squares.
// All reductions are deterministic: fixed grids, per-block partials in a
// fixed order, integer atomics only.
#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>

#include "pms_internal.h"

namespace pms {
namespace {

constexpr int kT = 256;

__device__ __forceinline__ bool pred_off(const int* pred) { return pred && *pred == 0; }

// ----------------------------------------------------------------------------- copies
// Streaming copy/fill: 16-byte accesses, four per thread in flight, for the 16-byte-aligned bulk
// (the host checks alignment); the last n % 4 elements elementwise.
__global__ __launch_bounds__(kT) void k_copy(const float* __restrict__ src, float* __restrict__ dst, size_t n,
                                             const int* pred) {
  if (pred_off(pred)) return;
  const size_t n4 = n >> 2;
  const float4* __restrict__ s4 = reinterpret_cast<const float4*>(src);
  float4* __restrict__ d4 = reinterpret_cast<float4*>(dst);
  const size_t stride = (size_t)gridDim.x * kT;
  size_t i = blockIdx.x * (size_t)kT + threadIdx.x;
  for (; i + 3 * stride < n4; i += 4 * stride) {
    const float4 a = s4[i], b = s4[i + stride], c = s4[i + 2 * stride], d = s4[i + 3 * stride];
    d4[i] = a;
    d4[i + stride] = b;
    d4[i + 2 * stride] = c;
    d4[i + 3 * stride] = d;
  }
  for (; i < n4; i += stride) d4[i] = s4[i];
  for (size_t t = (n4 << 2) + blockIdx.x * (size_t)kT + threadIdx.x; t < n; t += stride) dst[t] = src[t];
}

template <class T>
__global__ void k_copy1(const T* __restrict__ src, T* __restrict__ dst, size_t n, const int* pred) {
  if (pred_off(pred)) return;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

// n elements of a 4-byte type, p 16-byte aligned
template <class T>
__global__ __launch_bounds__(kT) void k_fill16(T* __restrict__ p, size_t n, T v) {
  const size_t n4 = n >> 2;
  uint4 w;
  w.x = w.y = w.z = w.w = *reinterpret_cast<const uint32_t*>(&v);
  uint4* __restrict__ p4 = reinterpret_cast<uint4*>(p);
  const size_t stride = (size_t)gridDim.x * kT;
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < n4; i += stride) p4[i] = w;
  for (size_t t = (n4 << 2) + blockIdx.x * (size_t)kT + threadIdx.x; t < n; t += stride) p[t] = v;
}

template <class T>
__global__ void k_masked_copy(const T* __restrict__ src, const uint8_t* __restrict__ m, T* __restrict__ dst, size_t n,
                              const int* pred) {
  if (pred_off(pred)) return;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = m[i] ? src[i] : (T)0;
}

__global__ void k_fill_f32(float* p, size_t n, float v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

__global__ void k_fill_u32(uint32_t* p, size_t n, uint32_t v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

// dst (n x n) = src window [r0, r0+n) x [c0, c0+n) of a (ld-wide) plane, optional multiply by mask window
template <class T, class TIN>
__global__ void k_window(const TIN* __restrict__ src, int ld, int r0, int c0, int n, const T* __restrict__ mul,
                         T* __restrict__ dst) {
  const size_t tot = (size_t)n * n;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < tot; i += (size_t)gridDim.x * blockDim.x) {
    const int r = (int)(i / n), c = (int)(i % n);
    const size_t s = (size_t)(r0 + r) * ld + (c0 + c);
    T v = (T)src[s];
    if (mul) v *= mul[s];
    dst[i] = v;
  }
}

// ----------------------------------------------------------------------------- MAD median
struct Rect {
  int r0, r1, c0, c1;  // [r0, r1) x [c0, c1)
};

__device__ __forceinline__ bool in_noise_mask(int r, int c, Rect inc, Rect exc) {
  const bool in = r >= inc.r0 && r < inc.r1 && c >= inc.c0 && c < inc.c1;
  const bool ex = r >= exc.r0 && r < exc.r1 && c >= exc.c0 && c < exc.c1;
  return in && !ex;
}

// Sort keys of |w|: the bits of a non-negative float (or double) order like an unsigned integer.
template <class T>
struct MadKey;
template <>
struct MadKey<float> {
  using K = uint32_t;
  __device__ static K key(float v) { return __float_as_uint(v) & 0x7fffffffu; }
  __device__ static float val(K k) { return __uint_as_float(k); }
};
template <>
struct MadKey<double> {
  using K = unsigned long long;
  __device__ static K key(double v) { return (K)__double_as_longlong(v) & 0x7fffffffffffffffull; }
  __device__ static double val(K k) { return __longlong_as_double((long long)k); }
};

// per-plane select state of the radix select
struct alignas(16) SelState {
  uint32_t prefix;   // fixed high bits of the target key
  uint32_t hi_key;   // min key above the low median (for even counts)
  uint32_t rank;     // remaining rank of the low median inside the prefix bucket
  uint32_t eq;       // count of keys equal to the final low median
  uint32_t n;        // number of keys
};
constexpr size_t kSelBytes = 32;
static_assert(sizeof(SelState) <= kSelBytes, "select state exceeds its slot");

constexpr int kBins = 2048;
constexpr int kMaxPlanes = 16;  // plane stacks handled per call (scale counts up to 16)

// Histogram of one digit of the keys whose higher digits equal the prefix found so far.  With
// `above` set (the last digit), keys whose higher digits exceed the prefix are all larger than the
// low median: the smallest of them goes to hi_key (atomic min), where the last select finds it if
// the low median's bucket holds no larger key (the successor of even counts, without a pass of its own).
template <bool MASKED>
__global__ __launch_bounds__(kT) void k_mad_hist(const float* __restrict__ planes, size_t plane, int w, Rect inc,
                                                 Rect exc, int shift, int nbits, int prefix_shift, int above,
                                                 SelState* __restrict__ st, uint32_t* __restrict__ hist,
                                                 const int* pred) {
  using K = uint32_t;
  if (pred_off(pred)) return;
  __shared__ uint32_t h[kBins];
  const int s = blockIdx.y;
  for (int i = threadIdx.x; i < kBins; i += kT) h[i] = 0;
  __syncthreads();
  const float* x = planes + (size_t)s * plane;
  const K pre = st[s].prefix;
  const K dmask = ((K)1 << nbits) - 1;
  const K none = ~(K)0;
  K best = none;
  auto add = [&](float v) {
    const K key = MadKey<float>::key(v);
    if (prefix_shift < 32) {
      const K kp = key >> prefix_shift, pp = pre >> prefix_shift;
      if (kp != pp) {
        if (above && kp > pp && key < best) best = key;
        return;
      }
    }
    atomicAdd(&h[(uint32_t)((key >> shift) & dmask)], 1u);
  };
  const size_t stride = (size_t)gridDim.x * kT;
  if (!MASKED && (reinterpret_cast<uintptr_t>(x) & 15) == 0) {
    // eight keys per thread and iteration, loaded as two float4 before any histogram update, so a
    // thread has two loads in flight instead of one per atomic (the counts do not depend on order)
    const float4* x4 = reinterpret_cast<const float4*>(x);
    const size_t n4 = plane >> 2;
    size_t i = blockIdx.x * (size_t)kT + threadIdx.x;
    for (; i + stride < n4; i += 2 * stride) {
      const float4 a = x4[i], b = x4[i + stride];
      add(a.x), add(a.y), add(a.z), add(a.w), add(b.x), add(b.y), add(b.z), add(b.w);
    }
    if (i < n4) {
      const float4 a = x4[i];
      add(a.x), add(a.y), add(a.z), add(a.w);
    }
    for (size_t j = 4 * n4 + blockIdx.x * (size_t)kT + threadIdx.x; j < plane; j += stride) add(x[j]);
  } else {
    for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < plane; i += stride) {
      if (MASKED) {
        const int r = (int)(i / w), c = (int)(i % w);
        if (!in_noise_mask(r, c, inc, exc)) continue;
      }
      add(x[i]);
    }
  }
  __syncthreads();
  uint32_t* gh = hist + (size_t)s * kBins;
  for (int i = threadIdx.x; i < kBins; i += kT)
    if (h[i]) atomicAdd(&gh[i], h[i]);
  if (above) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const K v = __shfl_xor(best, o, 64);
      best = v < best ? v : best;
    }
    // one atomic per block (per-wave atomics on the one address serialise at the L2)
    __shared__ K wmin[kT / 64];
    if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int k = 1; k < kT / 64; ++k) best = wmin[k] < best ? wmin[k] : best;
      if (best != none) atomicMin(&st[s].hi_key, best);
    }
  }
}

// one block per plane: locate the bucket holding the target rank, extend the prefix, clear the histogram
__global__ __launch_bounds__(kT) void k_mad_select(SelState* st, uint32_t* hist, int shift, int nbits, int last,
                                                   const int* pred) {
  using K = uint32_t;
  if (pred_off(pred)) return;
  const int s = blockIdx.x;
  uint32_t* gh = hist + (size_t)s * kBins;
  __shared__ uint32_t cnt[kBins];
  __shared__ uint32_t part[kT];
  const int nb = 1 << nbits;
  const int per = kBins / kT;  // 8 bins per thread
  const SelState S0 = st[s];  // read by every thread before the barrier; one thread writes it after
  uint32_t local = 0;
  for (int k = 0; k < per; ++k) {
    const int b = threadIdx.x * per + k;
    const uint32_t v = (b < nb) ? gh[b] : 0u;
    cnt[b] = v;
    local += v;
    gh[b] = 0u;
  }
  // inclusive scan of the per-thread counts (wave shuffles, then the wave totals)
  uint32_t inc = local;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t v = __shfl_up(inc, o, 64);
    if (lane >= o) inc += v;
  }
  if (lane == 63) part[wid] = inc;
  __syncthreads();
  uint32_t before = 0;
  for (int k = 0; k < wid; ++k) before += part[k];
  inc += before;
  const uint32_t exc = inc - local;
  // the thread whose range of ranks [exc, inc) holds the target rank finishes the search (the
  // last thread also takes a rank beyond the total, as the serial scan did)
  const bool mine = (S0.rank >= exc && S0.rank < inc) || (threadIdx.x == kT - 1 && S0.rank >= inc);
  __shared__ SelState s_state;
  __shared__ int s_bin;
  if (mine) {
    SelState S = S0;
    uint32_t run = exc;
    const int t = threadIdx.x;
    int b = t * per;
    for (; b < t * per + per - 1; ++b) {
      if (run + cnt[b] > S.rank) break;
      run += cnt[b];
    }
    S.rank -= run;
    S.prefix |= (K)b << shift;
    if (last) S.eq = cnt[b];
    s_state = S;
    s_bin = b;
  }
  __syncthreads();
  if (!last) {
    if (threadIdx.x == 0) st[s] = s_state;
    return;
  }
  // the smallest key above the low median: the next non-empty bucket of this last digit (same
  // higher digits), else the smallest key with larger higher digits (hi_key, from the histogram pass)
  const int b = s_bin;
  int nxt = kBins;
  for (int k = 0; k < per; ++k) {
    const int bb = threadIdx.x * per + k;
    if (bb > b && bb < nb && cnt[bb] != 0u && bb < nxt) nxt = bb;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const int v = __shfl_xor(nxt, o, 64);
    nxt = v < nxt ? v : nxt;
  }
  __shared__ int s_nxt[kT / 64];
  if (lane == 0) s_nxt[wid] = nxt;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kT / 64; ++k) nxt = s_nxt[k] < nxt ? s_nxt[k] : nxt;
    SelState S = s_state;
    const K dm = (((K)1 << nbits) - 1) << shift;  // this digit's bits
    if (nxt < nb) S.hi_key = (S.prefix & ~dm) | ((K)nxt << shift);
    st[s] = S;
  }
}

__global__ void k_mad_init(SelState* st, int S, uint32_t n) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  SelState z{};
  z.n = n;
  z.rank = (n - 1) / 2;
  z.prefix = 0;
  z.hi_key = ~0u;  // lowered by the last histogram pass and the last select
  st[s] = z;
}

__global__ void k_mad_finish(const SelState* st, int S, double* thr, const int* pred) {
  if (pred_off(pred)) return;
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  const SelState z = st[s];
  const uint32_t klo = (z.n - 1) / 2;
  const float vlo = MadKey<float>::val(z.prefix);
  double med = (double)vlo;
  if ((z.n & 1u) == 0) {
    // rank of the last key equal to vlo = first + eq - 1, first = klo - remaining rank
    const uint32_t first = klo - z.rank;
    const uint32_t lastr = first + z.eq - 1;
    const float vhi = (klo + 1 <= lastr) ? vlo : MadKey<float>::val(z.hi_key);
    med = ((double)vlo + (double)vhi) * 0.5;
  }
  thr[s] = med / 0.6745;
}

// four plane elements, read or stored together where the alignment allows
template <class T>
struct alignas(16) Quad {
  T a[4];
};
// stored past the caches, 16 bytes at a time
template <class T>
__device__ __forceinline__ void store_stream(T* p, const Quad<T>& q) {
  constexpr int N = 16 / (int)sizeof(T);
  typedef T V __attribute__((ext_vector_type(N)));
#pragma unroll
  for (int k = 0; k < 4 / N; ++k) {
    V v;
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = q.a[k * N + i];
    __builtin_nontemporal_store(v, reinterpret_cast<V*>(p) + k);
  }
}

// ---- median in one reading of the planes -------------------------------------------------------
// The radix select above (float32, for callers without a workspace and planes of 2^32 pixels) reads a plane once per
// digit.  With a workspace for it, a plane is read once:
//   * planes of at most 32768 noise pixels are selected by one block with the keys in registers;
//   * larger ones are sampled (k_mad_pivot: one block a plane, a radix select on the sample) for a range of
//     keys [lo, lo + range] around the median.  The sample is groups of four neighbours; were the four
//     always alike, the range would still reach four standard deviations of the median's rank to
//     either side.  One pass over the plane (k_mad_scan) counts the keys below the range, counts those in
//     it in 64 bins and sets them aside (6 to 9% of the plane), and one block a plane (k_mad_pick) takes the
//     bin of the median's rank and selects in it (from a list of that bin, k_mad_collect, on large planes).
// An end of the range that many keys are equal to (blanked pixels, quantised values) is not a part of it: those keys
// are only counted, so that the range holds what the sample says of it whatever the values (see MadRange::tied).
// Nothing is estimated in the result: when the range misses the median's rank or more keys fall in it
// than there is room for, k_mad_pick selects from the plane itself, with one block; the sample all but rules that
// out.  The result is the same key, and for even counts the same pair of keys, as the radix select's.
constexpr int kMT = 1024;            // threads of the one-block kernels
constexpr int kMadOne = 32 * kMT;    // noise pixels that one block holds in registers
constexpr int kMadBins = 64;         // bins of the range

// tied: the sample's ends of the range are the keys lo - 1 and lo + range + 1, outside it and counted by themselves.
// Such a range often starts at the smallest denormal (above zeros) and spans many binades, so its bins are of equal
// width in value, not in key: bins of equal key width put half of it in one (seven 4096^2 planes with 48% zeros: 520 us).
template <class K>
struct alignas(16) MadRange {
  K lo, range;      // keys lo .. lo + range (inclusive)
  K least2;         // k_mad_collect: least key of the successor's bin
  uint32_t shift;   // bin = (key - lo) >> shift, below kMadBins; tied: bits of `range`, bin = tied_bin(key)
  uint32_t tied;
  float scale;      // tied: kMadBins / (value of the upper end - value of lo)
  uint32_t at_lo;   // tied: keys equal to lo - 1
  uint32_t at_hi;   // tied: keys equal to lo + range + 1
  uint32_t below;   // keys below lo
  uint32_t n;       // keys of the range set aside (counted beyond the room for them)
  uint32_t listed;  // k_mad_collect: keys of the median's bin (counted beyond the room for them)
};
constexpr size_t kRangeBytes = 64;
static_assert(sizeof(MadRange<uint32_t>) <= kRangeBytes && sizeof(MadRange<unsigned long long>) <= kRangeBytes,
              "median range exceeds its slot");

// keys set aside per plane at most (a multiple of 16: each plane's buffer starts 64-byte aligned)
__host__ __device__ __forceinline__ size_t mad_room(size_t plane) { return (plane / 8 / 16 + 64) * 16; }
// keys of the median's bin listed per plane at most
__host__ __device__ __forceinline__ size_t mad_list_room(size_t plane) { return plane / 128 + 4096; }

template <class K>
__device__ __forceinline__ int bit_length(K v) {
  if constexpr (sizeof(K) == 8)
    return v ? 64 - __clzll((long long)v) : 0;
  else
    return v ? 32 - __clz((int)v) : 0;
}

// Bin of a key of a tied range whose least value is `low`.  Each operation is monotonic and a NaN (an infinite or NaN
// end) comes out alike for all keys, so the bins are in the keys' order whatever the scale.
template <class T>
__device__ __forceinline__ int tied_bin(typename MadKey<T>::K key, T low, float scale) {
  const T x = (MadKey<T>::val(key) - low) * (T)scale;
  return x < (T)(kMadBins - 1) ? (int)x : kMadBins - 1;
}

// Where a block finds ranks in the 2048 counts of h (LDS): the bin, the counts before it and its own.
// All threads of a kMT block call it; the result is the same in all of them.  A rank beyond the total
// gives the last bin.
struct BinHit {
  int bin;
  uint32_t before, count;
};
struct BinScratch {
  uint32_t part[kMT / 64];
  BinHit hit[2];
};
__device__ __forceinline__ void find_bins(const uint32_t* h, uint32_t r0, uint32_t r1, BinScratch& sc, BinHit* a,
                                          BinHit* b) {
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  const uint32_t c0 = h[2 * t], c1 = h[2 * t + 1], local = c0 + c1;
  uint32_t inc = local;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t v = __shfl_up(inc, o, 64);
    if (lane >= o) inc += v;
  }
  __syncthreads();  // the scratch of an earlier call has been read
  if (lane == 63) sc.part[wid] = inc;
  __syncthreads();
  uint32_t before = lane < wid ? sc.part[lane & (kMT / 64 - 1)] : 0;  // lanes 0 .. 15 hold the waves before
#pragma unroll
  for (int o = kMT / 128; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
  inc += (uint32_t)__builtin_amdgcn_readfirstlane((int)before);
  const uint32_t exc = inc - local;
  auto put = [&](uint32_t r, BinHit* to) {
    if ((r >= exc && r < inc) || (t == kMT - 1 && r >= inc)) {
      const bool second = r >= exc + c0;
      *to = BinHit{2 * t + (second ? 1 : 0), second ? exc + c0 : exc, second ? c1 : c0};
    }
  };
  put(r0, &sc.hit[0]);
  put(r1, &sc.hit[1]);
  __syncthreads();
  *a = sc.hit[0];
  *b = sc.hit[1];
}
__device__ __forceinline__ BinHit find_bin(const uint32_t* h, uint32_t r, BinScratch& sc) {
  BinHit a, b;
  find_bins(h, r, r, sc, &a, &b);
  return a;
}

__device__ __forceinline__ void clear_bins(uint32_t* h) {
  h[threadIdx.x] = 0;
  h[threadIdx.x + kMT] = 0;
}

// minimum over a kMT block, the same in all threads
template <class K>
__device__ __forceinline__ K block_min_key(K v, K* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const K u = __shfl_xor(v, o, 64);
    v = u < v ? u : v;
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  for (int k = 0; k < kMT / 64; ++k) v = red[k] < v ? red[k] : v;
  return v;
}

template <class T>
__device__ __forceinline__ double mad_of(typename MadKey<T>::K lo, typename MadKey<T>::K hi, bool even) {
  const double a = (double)MadKey<T>::val(lo);
  return (even ? (a + (double)MadKey<T>::val(hi)) * 0.5 : a) / 0.6745;
}

// The key of noise pixel j of a plane in the order of the included rectangle's rows (the whole plane
// without a mask); false for a pixel of the excluded rectangle.
template <class T, bool MASKED>
__device__ __forceinline__ bool noise_key(const T* x, int w, Rect inc, Rect exc, uint32_t j,
                                          typename MadKey<T>::K* key) {
  if constexpr (!MASKED) {
    *key = MadKey<T>::key(x[j]);
    return true;
  } else {
    const uint32_t wr = (uint32_t)(inc.c1 - inc.c0);
    const uint32_t q = j / wr;
    const int r = inc.r0 + (int)q, c = inc.c0 + (int)(j - q * wr);
    *key = MadKey<T>::key(x[(size_t)r * w + c]);
    return !(r >= exc.r0 && r < exc.r1 && c >= exc.c0 && c < exc.c1);
  }
}

// Every noise pixel's key of a plane, dealt over `nthr` threads, to f(key).
template <class T, bool MASKED, class F>
__device__ __forceinline__ void each_noise_key(const T* x, size_t plane, int w, Rect inc, Rect exc, size_t thr,
                                               size_t nthr, F f) {
  if constexpr (!MASKED) {
    constexpr int V = 16 / sizeof(T);
    struct alignas(16) Vec {
      T a[V];
    };
    size_t done = 0;
    if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {
      const Vec* xv = reinterpret_cast<const Vec*>(x);
      const size_t nv = plane / V;
      size_t i = thr;
      for (; i + 3 * nthr < nv; i += 4 * nthr) {  // four loads in flight
        const Vec a = xv[i], b = xv[i + nthr], c = xv[i + 2 * nthr], d = xv[i + 3 * nthr];
#pragma unroll
        for (int k = 0; k < V; ++k) f(MadKey<T>::key(a.a[k]));
#pragma unroll
        for (int k = 0; k < V; ++k) f(MadKey<T>::key(b.a[k]));
#pragma unroll
        for (int k = 0; k < V; ++k) f(MadKey<T>::key(c.a[k]));
#pragma unroll
        for (int k = 0; k < V; ++k) f(MadKey<T>::key(d.a[k]));
      }
      for (; i < nv; i += nthr) {
        const Vec a = xv[i];
#pragma unroll
        for (int k = 0; k < V; ++k) f(MadKey<T>::key(a.a[k]));
      }
      done = nv * V;
    }
    for (size_t i = done + thr; i < plane; i += nthr) f(MadKey<T>::key(x[i]));
  } else {
    // 64 threads a row: no division per pixel
    const int lane = (int)(thr & 63);
    for (size_t r = inc.r0 + (thr >> 6); r < (size_t)inc.r1; r += nthr >> 6) {
      const T* row = x + r * w;
      const bool cut = (int)r >= exc.r0 && (int)r < exc.r1;
      for (int c = inc.c0 + lane; c < inc.c1; c += 64) {
        if (cut && c >= exc.c0 && c < exc.c1) continue;
        f(MadKey<T>::key(row[c]));
      }
    }
  }
}

// Whole planes of at most kMadOne noise pixels (area: pixels of the included rectangle): a radix select
// in LDS over keys held in registers, 11 bits a digit; then the successor of an even count.
template <class T, bool MASKED, int PT>
__global__ __launch_bounds__(kMT) void k_mad_one(const T* __restrict__ planes, size_t plane, int w, Rect inc, Rect exc,
                                                 uint32_t area, uint32_t count, double* __restrict__ thr,
                                                 const int* pred) {
  using K = typename MadKey<T>::K;
  if (pred_off(pred)) return;
  __shared__ uint32_t h[kBins];
  __shared__ BinScratch scratch;
  __shared__ K red[kMT / 64];
  const T* x = planes + (size_t)blockIdx.x * plane;
  K key[PT];
  uint32_t have = 0;
#pragma unroll
  for (int i = 0; i < PT; ++i) {
    const uint32_t j = threadIdx.x + i * kMT;
    const bool in = noise_key<T, MASKED>(x, w, inc, exc, min(j, area - 1), &key[i]);
    if (in && j < area) have |= 1u << i;
  }
  uint32_t rank = (count - 1) / 2;  // of the low median among the keys that share the digits found so far
  K v = 0;
  int top = 8 * (int)sizeof(K) - 1;  // the sign bit is clear
  uint32_t equal = count;
  while (top > 0) {
    const int nd = min(11, top), shift = top - nd;
    clear_bins(h);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PT; ++i)
      if ((have >> i) & 1 && (key[i] >> top) == (v >> top))
        atomicAdd(&h[(uint32_t)(key[i] >> shift) & ((1u << nd) - 1)], 1u);
    __syncthreads();
    const BinHit b = find_bin(h, rank, scratch);
    v |= (K)b.bin << shift;
    rank -= b.before;
    equal = b.count;
    top = shift;
  }
  const bool even = (count & 1) == 0;
  K hi = v;
  if (even && rank + 1 >= equal) {
    K m = ~(K)0;
#pragma unroll
    for (int i = 0; i < PT; ++i)
      if ((have >> i) & 1 && key[i] > v && key[i] < m) m = key[i];
    hi = block_min_key(m, red);
  }
  if (threadIdx.x == 0) thr[blockIdx.x] = mad_of<T>(v, hi, even);
}

// Sampled range of keys around the median; also clears the plane's counters and bins.  PT keys a
// thread, four neighbours from each of the sample's strata (one cache line each) at a place that a
// hash picks, so that a pattern in the plane does not line up with them.
template <class T, bool MASKED, int PT>
__global__ __launch_bounds__(kMT) void k_mad_pivot(const T* __restrict__ planes, size_t plane, int w, Rect inc,
                                                   Rect exc, uint32_t area, MadRange<typename MadKey<T>::K>* st,
                                                   uint32_t* __restrict__ hist, const int* pred) {
  using K = typename MadKey<T>::K;
  if (pred_off(pred)) return;
  constexpr int kKeyBits = 8 * sizeof(K) - 1;
  __shared__ uint32_t h0[kBins], h1[kBins];
  __shared__ BinScratch scratch;
  __shared__ K red[kMT / 64];
  __shared__ uint32_t taken;
  const int s = blockIdx.x, t = threadIdx.x;
  const T* x = planes + (size_t)s * plane;
  if (t < kMadBins) hist[(size_t)s * kMadBins + t] = 0;
  if (t == 0) taken = 0;
  const uint32_t stratum = area / (PT / 4 * kMT);  // at least 16 (area > kMadOne)
  const auto sample = [&](const T* from, K(&key)[PT]) {  // returns which of the keys are noise pixels'
    uint32_t have = 0;
    const bool vec = !MASKED && (reinterpret_cast<uintptr_t>(from) & 15) == 0;
#pragma unroll
    for (int i = 0; i < PT / 4; ++i) {
      const uint32_t c = t + i * kMT;
      const uint32_t at = c * stratum + ((c * 2654435761u) >> 8) % (stratum - 3);
      if (vec) {
        const Quad<T> q = reinterpret_cast<const Quad<T>*>(from)[at / 4];
#pragma unroll
        for (int k = 0; k < 4; ++k) key[4 * i + k] = MadKey<T>::key(q.a[k]);
        have |= 15u << (4 * i);
        continue;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (noise_key<T, MASKED>(from, w, inc, exc, at + k, &key[4 * i + k])) have |= 1u << (4 * i + k);
    }
    return have;
  };
  K key[PT];
  const uint32_t have = sample(x, key);
  __syncthreads();
  atomicAdd(&taken, (uint32_t)__popc(have));
  __syncthreads();
  const uint32_t m = taken;
  const uint32_t half = (uint32_t)(4.f * sqrtf((float)m)) + 8;
  uint32_t r0 = m / 2 > half ? m / 2 - half : 0, r1 = m / 2 + half;
  const bool open0 = m / 2 <= half, open1 = r1 >= m;
  // Digits of both ends: two, which is a range's width to better than a tenth, and more while over 1/128 of the
  // sample shares an end's digits and not its value: with the 1/15 of the sample between the ends (1/11 of 8192
  // keys) the range then stays within the room for it, 1/8, once an end that many keys are equal to is not in it.
  K lo = 0, hi = 0;
  uint32_t n_lo = 0, n_hi = 0;  // keys that share an end's digits
  const auto digit = [&](const K(&q)[PT], uint32_t live, int top) {  // the one below bit `top`
    const int nd = min(11, top), shift = top - nd;
    const bool apart = lo != hi;
    clear_bins(h0);
    clear_bins(h1);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      if (!((live >> i) & 1)) continue;
      const uint32_t d = (uint32_t)(q[i] >> shift) & ((1u << nd) - 1);
      if ((q[i] >> top) == (lo >> top)) atomicAdd(&h0[d], 1u);
      if (apart && (q[i] >> top) == (hi >> top)) atomicAdd(&h1[d], 1u);
    }
    __syncthreads();
    BinHit a, b;
    find_bins(h0, r0, r1, scratch, &a, &b);
    if (apart) b = find_bin(h1, r1, scratch);
    lo |= (K)a.bin << shift;
    hi |= (K)b.bin << shift;
    r0 -= a.before;
    r1 -= b.before;
    n_lo = a.count;
    n_hi = b.count;
  };
  int rest = kKeyBits;
  for (; rest > kKeyBits - 22; rest -= 11) digit(key, have, rest);
  const uint32_t few = m / 128;
  if (n_lo > few || n_hi > few) {
    // The sample is read again: kept in registers until here, it made the kernel 18 -> 22 us where nothing is tied.
    const T* again = x;
    asm volatile("" : "+s"(again));
    K q[PT];
    const uint32_t live = sample(again, q);
    // are the keys that share an end's digits one value?
    K least_lo = ~(K)0, high_lo = ~(K)0, least_hi = ~(K)0, high_hi = ~(K)0;  // high: complement of the greatest
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      if (!((live >> i) & 1)) continue;
      const K prefix = q[i] >> rest;
      if (prefix == (lo >> rest)) least_lo = min(least_lo, q[i]), high_lo = min(high_lo, ~q[i]);
      if (prefix == (hi >> rest)) least_hi = min(least_hi, q[i]), high_hi = min(high_hi, ~q[i]);
    }
    least_lo = block_min_key(least_lo, red);
    high_lo = ~block_min_key(high_lo, red);
    least_hi = block_min_key(least_hi, red);
    high_hi = ~block_min_key(high_hi, red);
    if ((n_lo <= few || least_lo == high_lo) && (n_hi <= few || least_hi == high_hi)) {
      lo = n_lo > few ? least_lo : lo;
      hi = n_hi > few ? least_hi : hi | (((K)1 << rest) - 1);
      rest = 0;
    } else {
      for (; rest > 0 && (n_lo > few || n_hi > few); rest = max(rest - 11, 0)) digit(q, live, rest);
    }
  }
  if (t == 0) {
    MadRange<K> z{};
    if (rest == 0 && hi - lo >= 2 && !open0 && !open1) {
      const K upper = hi--;
      z.tied = 1;
      ++lo;
      z.scale = (float)kMadBins / (float)(MadKey<T>::val(upper) - MadKey<T>::val(lo));
    }
    hi |= ((K)1 << rest) - 1;
    if (open0) lo = 0;
    if (open1) hi = ((K)1 << kKeyBits) - 1;
    z.lo = lo;
    z.range = hi - lo;
    z.least2 = ~(K)0;
    const int bits = bit_length<K>(z.range);
    z.shift = z.tied ? bits : bits > 6 ? bits - 6 : 0;
    st[s] = z;
  }
}

// The pass over the planes, eight keys (four float64) a thread at a time: keys below the range are
// counted, keys in it go to an LDS bin and to the wave's part of an LDS list (slots from a prefix sum
// over the wave, no atomic), which the wave appends to the plane's buffer with one reservation when it fills
// and at the end.  Bound: reading the planes (104 us for seven of 4096^2, against 95 us for each of the radix
// select's three passes); what stands above that is the prefix sums and bins.  A reservation for every few
// hundred keys of a wave made it 279 us: atomics on one address follow one another.  A tied range has a form
// of its own, which counts the ends' keys too.
template <class T, bool MASKED>
__global__ __launch_bounds__(kT) void k_mad_scan(const T* __restrict__ planes, size_t plane, int w, Rect inc, Rect exc,
                                                 MadRange<typename MadKey<T>::K>* __restrict__ st,
                                                 uint32_t* __restrict__ hist,
                                                 typename MadKey<T>::K* __restrict__ aside, size_t room,
                                                 const int* pred) {
  using K = typename MadKey<T>::K;
  if (pred_off(pred)) return;
  constexpr int V = 16 / sizeof(T), G = 2 * V;  // keys of a vector, of a group
  constexpr int kStage = 64 * G + 768;          // room for a large plane's share of a wave: one reservation a block
  __shared__ uint32_t h[kMadBins];
  __shared__ K stage[kT / 64][kStage];
  __shared__ uint32_t counts[kT / 64], belows[kT / 64], ends[2][kT / 64], base_all;
  const int s = blockIdx.y;
  MadRange<K>* S = st + s;
  const K lo = S->lo, range = S->range;
  const uint32_t shift = S->shift, tied = S->tied;
  K* out = aside + (size_t)s * room;
  if (threadIdx.x < kMadBins) h[threadIdx.x] = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  K* mine = stage[threadIdx.x >> 6];
  uint32_t below = 0, at_lo = 0, at_hi = 0;
  int n = 0;  // keys in the wave's part, the same in all its lanes
  auto flush = [&] {
    __builtin_amdgcn_wave_barrier();  // the other lanes' LDS writes precede the reads below (one wave: in order)
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(&S->n, (uint32_t)n);
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    for (int i = lane; i < n; i += 64)
      if ((size_t)base + i < room) out[base + i] = mine[i];
    n = 0;
    __builtin_amdgcn_wave_barrier();
  };
  const T low = MadKey<T>::val(lo);
  const float scale = S->scale;
  const auto pass = [&](auto tc) {
    constexpr bool TIED = decltype(tc)::value;
    // `live`: which of the lane's keys are noise pixels; every lane of a wave takes every group
    auto take = [&](const K (&key)[G], uint32_t live) {
      uint32_t in = 0;
#pragma unroll
      for (int k = 0; k < G; ++k) {
        below += (live >> k) & (key[k] < lo ? 1u : 0u);
        in |= key[k] - lo <= range ? 1u << k : 0u;
      }
      in &= live;
      if constexpr (TIED) {
#pragma unroll
        for (int k = 0; k < G; ++k) {
          at_lo += (live >> k) & (key[k] == lo - 1 ? 1u : 0u);
          at_hi += (live >> k) & (key[k] == lo + range + 1 ? 1u : 0u);
        }
      }
      uint32_t at = __popc(in);
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t v = __shfl_up(at, o, 64);
        if (lane >= o) at += v;
      }
      const int total = __builtin_amdgcn_readlane((int)at, 63);
      if (total == 0) return;
      at += (uint32_t)n - __popc(in);
#pragma unroll
      for (int k = 0; k < G; ++k) {
        if (!((in >> k) & 1)) continue;
        if constexpr (TIED)
          atomicAdd(&h[tied_bin<T>(key[k], low, scale)], 1u);
        else
          atomicAdd(&h[(uint32_t)((key[k] - lo) >> shift)], 1u);
        mine[at + __popc(in & ((1u << k) - 1))] = key[k];
      }
      if (shift != 0) n += total;  // otherwise a bin is one key and the bins say all
      if (n > kStage - 64 * G) flush();
    };
    const T* x = planes + (size_t)s * plane;
    const size_t thr = blockIdx.x * (size_t)kT + threadIdx.x, nthr = (size_t)gridDim.x * kT;
    K key[G];
    if constexpr (!MASKED) {
      struct alignas(16) Vec {
        T a[V];
      };
      const size_t nv = (reinterpret_cast<uintptr_t>(x) & 15) == 0 ? plane / V : 0;
      const Vec* xv = reinterpret_cast<const Vec*>(x);
      for (size_t i0 = thr - lane; i0 < nv; i0 += 2 * nthr) {  // the wave's first vector
        uint32_t live = 0;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const size_t i = i0 + u * nthr + lane;
          const Vec v = xv[min(i, nv - 1)];
          live |= i < nv ? ((1u << V) - 1) << (u * V) : 0u;
#pragma unroll
          for (int k = 0; k < V; ++k) key[u * V + k] = MadKey<T>::key(v.a[k]);
        }
        take(key, live);
      }
      for (size_t i0 = nv * V + thr - lane; i0 < plane; i0 += G * nthr) {
        uint32_t live = 0;
#pragma unroll
        for (int k = 0; k < G; ++k) {
          const size_t i = i0 + k * nthr + lane;
          key[k] = MadKey<T>::key(x[min(i, plane - 1)]);
          live |= i < plane ? 1u << k : 0u;
        }
        take(key, live);
      }
    } else {
      // a wave takes two rows by G / 2 columns a lane: no division per pixel
      const int rstep = (int)(nthr >> 6);
      for (int r = inc.r0 + (int)(thr >> 6); r < inc.r1; r += 2 * rstep) {
        for (int c0 = inc.c0 + lane; c0 - lane < inc.c1; c0 += 32 * G) {
          uint32_t live = 0;
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int y = r + u * rstep;
            const T* row = x + (size_t)min(y, inc.r1 - 1) * w;
            const bool cut = y >= exc.r0 && y < exc.r1;
#pragma unroll
            for (int k = 0; k < G / 2; ++k) {
              const int c = c0 + 64 * k;
              key[u * (G / 2) + k] = MadKey<T>::key(row[min(c, inc.c1 - 1)]);
              if (y < inc.r1 && c < inc.c1 && !(cut && c >= exc.c0 && c < exc.c1)) live |= 1u << (u * (G / 2) + k);
            }
          }
          take(key, live);
        }
      }
    }
  };
  tied ? pass(std::true_type{}) : pass(std::false_type{});
  // the block's remainder in one reservation: atomics on one address cost more than the copy
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) below += __shfl_xor(below, o, 64);
  if (tied) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      at_lo += __shfl_xor(at_lo, o, 64);
      at_hi += __shfl_xor(at_hi, o, 64);
    }
  }
  if (lane == 0) {
    counts[threadIdx.x >> 6] = (uint32_t)n;
    belows[threadIdx.x >> 6] = below;
    ends[0][threadIdx.x >> 6] = at_lo;
    ends[1][threadIdx.x >> 6] = at_hi;
  }
  __syncthreads();
  uint32_t before = 0, all = 0, less = 0;
  for (int k = 0; k < kT / 64; ++k) {
    before += k < (int)(threadIdx.x >> 6) ? counts[k] : 0;
    all += counts[k];
    less += belows[k];
  }
  if (threadIdx.x == 0) {
    base_all = all ? atomicAdd(&S->n, all) : 0;
    if (less) atomicAdd(&S->below, less);
  }
  if (tied && threadIdx.x < 2) {
    uint32_t v = 0;
    for (int k = 0; k < kT / 64; ++k) v += ends[threadIdx.x][k];
    if (v) atomicAdd(threadIdx.x ? &S->at_hi : &S->at_lo, v);
  }
  if (threadIdx.x < kMadBins && h[threadIdx.x])
    atomicAdd(&hist[(size_t)s * kMadBins + threadIdx.x], h[threadIdx.x]);
  __syncthreads();
  const size_t to = (size_t)base_all + before;
  for (int i = lane; i < n; i += 64)
    if (to + i < room) out[to + i] = mine[i];
}

// the 64 bins of a plane as the counts that find_bins takes
__device__ __forceinline__ void load_bins(uint32_t* h, const uint32_t* __restrict__ hist, int s) {
  clear_bins(h);
  if (threadIdx.x < kMadBins) h[threadIdx.x] = hist[(size_t)s * kMadBins + threadIdx.x];
  __syncthreads();
}

// Large planes: the keys of the median's bin and the least key of its successor's, by many blocks.
template <class T>
__global__ __launch_bounds__(kMT) void k_mad_collect(uint32_t count, MadRange<typename MadKey<T>::K>* __restrict__ st,
                                                     const uint32_t* __restrict__ hist,
                                                     const typename MadKey<T>::K* __restrict__ aside, size_t room,
                                                     typename MadKey<T>::K* __restrict__ lists, size_t list_room,
                                                     const int* pred) {
  using K = typename MadKey<T>::K;
  if (pred_off(pred)) return;
  __shared__ uint32_t h[kBins];
  __shared__ BinScratch scratch;
  constexpr int V = 16 / sizeof(K);
  __shared__ K stage[V * kMT];
  __shared__ uint32_t n_stage, base;
  const int s = blockIdx.y, t = threadIdx.x;
  MadRange<K>* S = st + s;
  const K lo = S->lo;
  const uint32_t shift = S->shift, tied = S->tied, below = S->below, n = S->n, k = (count - 1) / 2;
  const T low = MadKey<T>::val(lo);
  const float scale = S->scale;
  if (shift == 0 || n > room || k < below) return;
  load_bins(h, hist, s);
  BinHit b, b2;  // of ranks in the range; k_mad_pick finds out if they are not
  find_bins(h, k - below, k - below + ((count & 1) == 0 ? 1 : 0), scratch, &b, &b2);
  struct alignas(16) Vec {
    K a[V];
  };
  const Vec* bv = reinterpret_cast<const Vec*>(aside + (size_t)s * room);
  K* list = lists + (size_t)s * list_room;
  const uint32_t nv = (n + V - 1) / V;
  K least2 = ~(K)0;
  for (uint32_t i0 = blockIdx.x * kMT; i0 < nv; i0 += gridDim.x * kMT) {
    const uint32_t i = i0 + t;
    const Vec v = bv[min(i, nv - 1)];
    if (t == 0) n_stage = 0;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < V; ++e) {
      if (i >= nv || i * V + e >= n) break;
      const int bin = tied ? tied_bin<T>(v.a[e], low, scale) : (int)((v.a[e] - lo) >> shift);
      if (bin == b.bin)
        stage[atomicAdd(&n_stage, 1u)] = v.a[e];
      else if (bin == b2.bin)
        least2 = v.a[e] < least2 ? v.a[e] : least2;
    }
    __syncthreads();
    const uint32_t m = n_stage;
    if (t == 0 && m) base = atomicAdd(&S->listed, m);
    __syncthreads();
    for (uint32_t q = t; q < m; q += kMT)
      if ((size_t)base + q < list_room) list[base + q] = stage[q];
  }
  __shared__ K red[kMT / 64];
  least2 = block_min_key(least2, red);
  if (t == 0 && least2 != ~(K)0) atomicMin(&S->least2, least2);
}

// The median's rank in the bins, then digits of 11 bits of its bin's keys: from the list that k_mad_collect left
// (lists, large planes), from the keys set aside (the bin's gathered in LDS first where many digits are to come
// and they fit), or from the plane where the range missed the rank or its keys found no room.  A rank on a tied
// range's end needs no digits, nor does a tied range's bin of one value.
template <class T, bool MASKED>
__global__ __launch_bounds__(kMT) void k_mad_pick(const T* __restrict__ planes, size_t plane, int w, Rect inc, Rect exc,
                                                  uint32_t count,
                                                  const MadRange<typename MadKey<T>::K>* __restrict__ st,
                                                  const uint32_t* __restrict__ hist,
                                                  const typename MadKey<T>::K* __restrict__ aside, size_t room,
                                                  const typename MadKey<T>::K* __restrict__ lists, size_t list_room,
                                                  double* __restrict__ thr, const int* pred) {
  using K = typename MadKey<T>::K;
  if (pred_off(pred)) return;
  constexpr uint32_t kGather = 2048;
  __shared__ uint32_t h[kBins];
  __shared__ BinScratch scratch;
  __shared__ K red[kMT / 64];
  __shared__ K gathered[kGather];
  __shared__ uint32_t n_gathered;
  const int s = blockIdx.x, t = threadIdx.x;
  const T* x = planes + (size_t)s * plane;
  const MadRange<K> S = st[s];
  const K* const mine = aside + (size_t)s * room;
  const bool even = (count & 1) == 0;
  const uint32_t k = (count - 1) / 2, k2 = k + (even ? 1 : 0);
  load_bins(h, hist, s);
  const BinHit last = find_bin(h, 0xffffffffu, scratch);
  // f(key) of n keys, eight loads in flight
  const auto over = [&](const K* from, uint32_t n, auto f) {
    for (uint32_t i0 = t; i0 < n; i0 += 8 * kMT) {
      K q[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) q[u] = from[min(i0 + u * kMT, n - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (i0 + u * kMT < n) f(q[u]);
    }
  };
  // ranks of the range: S.below to above; S.at_lo ranks before and S.at_hi after are a tied range's ends
  const uint32_t above = S.below + last.before + last.count, end = above + S.at_hi;
  if (k2 < end && (k >= above || (k < S.below && k >= S.below - S.at_lo))) {
    const K v = k < S.below ? S.lo - 1 : S.lo + S.range + 1;
    K hi = v;
    if (k < S.below && k2 >= S.below) {  // the successor is the range's least key, or its upper end
      K m = S.lo + S.range + 1;
      if (above != S.below) {
        if (S.shift == 0)
          m = S.lo;  // the range is one key
        else if (S.n <= room)
          over(mine, S.n, [&](K key) { m = min(m, key); });
        else
          each_noise_key<T, MASKED>(x, plane, w, inc, exc, t, kMT, [&](K key) { m = key > v ? min(m, key) : m; });
      }
      hi = block_min_key(m, red);
    }
    if (t == 0) thr[s] = mad_of<T>(v, hi, even);
    return;
  }
  const bool found = k >= S.below && k < above && k2 < end;
  const bool set_aside = found && S.n <= room;
  const bool listed = set_aside && lists && S.listed <= list_room;
  const bool by_value = found && S.tied && S.shift != 0;
  // key - lo of every key that can be the median, and of at least all keys of the range up to its successor
  const K lo = found ? S.lo : 0;
  const T low = MadKey<T>::val(S.lo);
  K v = 0;
  K least2 = ~(K)0;
  uint32_t rank = k, equal = 0;
  int top = 8 * (int)sizeof(K) - 1;
  int bin = 0;
  bool only_bin = listed;  // the keys are the median's bin's, the successor's least is least2
  const K* from = listed ? lists + (size_t)s * list_room : mine;
  uint32_t n_from = listed ? S.listed : S.n;
  if (found) {
    BinHit b, b2;
    find_bins(h, k - S.below, k2 - S.below, scratch, &b, &b2);
    bin = b.bin;
    if (!S.tied) v = (K)bin << S.shift;
    rank = k - S.below - b.before;
    equal = b.count;
    top = (int)S.shift;
    const auto bin_of = [&](K key) { return by_value ? tied_bin<T>(key, low, S.scale) : (int)((key - lo) >> S.shift); };
    if (set_aside && !listed && top > 0 && equal <= kGather && (by_value || sizeof(K) == 8)) {
      if (t == 0) n_gathered = 0;
      __syncthreads();
      K m = ~(K)0;
      over(mine, S.n, [&](K key) {
        const int at = bin_of(key);
        if (at == bin)
          gathered[atomicAdd(&n_gathered, 1u)] = key;
        else if (at == b2.bin)
          m = min(m, key);
      });
      least2 = block_min_key(m, red) - lo;
      only_bin = true;
      from = gathered;
      n_from = equal;
    } else if (listed && b2.bin != bin) {
      least2 = S.least2 - lo;
    } else if (by_value && !listed) {
      // many keys in the bin: one value, or digits
      K m = ~(K)0, high = ~(K)0;  // the least key and the complement of the greatest
      const auto ends = [&](K key) {
        if (key < S.lo || key - S.lo > S.range || bin_of(key) != bin) return;
        m = min(m, key);
        high = min(high, ~key);
      };
      if (set_aside)
        over(mine, S.n, ends);
      else
        each_noise_key<T, MASKED>(x, plane, w, inc, exc, t, kMT, ends);
      m = block_min_key(m, red);
      high = ~block_min_key(high, red);
      if (m == high) {
        v = m - lo;
        top = 0;
      }
    }
    if (k2 >= above)
      least2 = S.range + 1;
    else if (S.shift == 0)
      least2 = (K)b2.bin;
  }
  auto each = [&](auto f) {
    if (only_bin || set_aside)
      over(from, n_from, [&](K key) { f(key - lo); });
    else
      each_noise_key<T, MASKED>(x, plane, w, inc, exc, t, kMT, [&](K key) {
        if (!found || key - lo <= S.range) f(key - lo);
      });
  };
  const auto digits = [&](auto tc) {
    while (top > 0) {
      const int nd = min(11, top), shift = top - nd;
      clear_bins(h);
      __syncthreads();
      each([&](K rel) {
        if ((rel >> top) != (v >> top)) return;
        const uint32_t d = (uint32_t)(rel >> shift) & ((1u << nd) - 1);
        if constexpr (decltype(tc)::value) {
          if (tied_bin<T>(rel + lo, low, S.scale) != bin) return;
          // one addition for all lanes with the first one's digit: equal keys would be added one after the other
          const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
          const unsigned long long same = __ballot(d == first);
          if (d != first)
            atomicAdd(&h[d], 1u);
          else if ((int)(t & 63) == __ffsll(same) - 1)
            atomicAdd(&h[d], (uint32_t)__popcll(same));
        } else {
          atomicAdd(&h[d], 1u);
        }
      });
      __syncthreads();
      const BinHit b = find_bin(h, rank, scratch);
      v |= (K)b.bin << shift;
      rank -= b.before;
      equal = b.count;
      top = shift;
    }
  };
  by_value && !only_bin ? digits(std::true_type{}) : digits(std::false_type{});
  K hi = v;
  if (even && rank + 1 >= equal) {
    K m = least2;
    if (!(found && S.shift == 0)) each([&](K rel) { m = rel > v && rel < m ? rel : m; });
    hi = block_min_key(m, red);
  }
  if (t == 0) thr[s] = mad_of<T>(lo + v, lo + hi, even);
}

// ----------------------------------------------------------------------------- threshold + maxima
// out = in where |in| > sigma * thr[s] (zero in the plane's border), and the outputs' maxima per block.
// k_threshold4: planes whose quads are aligned, four quads in flight a thread, STREAM: the output goes past the caches
// (launches that exceed them, see past_caches).  Bound: its bytes, 5.5 TB/s on seven 4096^2 planes: 171 us, 217 us one value at
// a time through the caches; the noise estimate that reads the input planes next finds more of them cached (142 -> 113 us).
template <class T, bool STREAM>
__global__ __launch_bounds__(kT) void k_threshold4(const T* __restrict__ in, T* __restrict__ out, size_t plane, int w,
                                                   const double* __restrict__ thr, double sigma,
                                                   const int* __restrict__ border, T* __restrict__ pmax,
                                                   const int* pred) {
  if (pred_off(pred)) return;
  const int s = blockIdx.y;
  const int h = (int)(plane / w);
  const double lim = sigma * thr[s];
  const int b = border ? border[s] : 0;
  const Quad<T>* x = reinterpret_cast<const Quad<T>*>(in + (size_t)s * plane);
  T* y = out + (size_t)s * plane;
  const size_t n4 = plane / 4;
  const size_t stride = (size_t)gridDim.x * kT;
  T m = -INFINITY;
  const auto one = [&](size_t i, const Quad<T>& v) {
    Quad<T> o;
#pragma unroll
    for (int k = 0; k < 4; ++k) o.a[k] = ((double)fabs(v.a[k]) > lim) ? v.a[k] : (T)0;
    if (border) {
      const int r = (int)(4 * i / w), c = (int)(4 * i % w);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (r < b || r >= h - b || c + k < b || c + k >= w - b) o.a[k] = 0;
    }
    if constexpr (STREAM)
      store_stream(y + 4 * i, o);
    else
      *reinterpret_cast<Quad<T>*>(y + 4 * i) = o;
#pragma unroll
    for (int k = 0; k < 4; ++k) m = o.a[k] > m ? o.a[k] : m;
  };
  size_t i = blockIdx.x * (size_t)kT + threadIdx.x;
  for (; i + 3 * stride < n4; i += 4 * stride) {  // four loads in flight
    const Quad<T> v0 = x[i], v1 = x[i + stride], v2 = x[i + 2 * stride], v3 = x[i + 3 * stride];
    one(i, v0);
    one(i + stride, v1);
    one(i + 2 * stride, v2);
    one(i + 3 * stride, v3);
  }
  for (; i < n4; i += stride) one(i, x[i]);
  m = block_max_t<T>(m);
  if (threadIdx.x == 0) pmax[(size_t)s * gridDim.x + blockIdx.x] = m;
}

// any other plane, a value at a time
template <class T>
__global__ __launch_bounds__(kT) void k_threshold(const T* __restrict__ in, T* __restrict__ out, size_t plane, int w,
                                                  const double* __restrict__ thr, double sigma,
                                                  const int* __restrict__ border, T* __restrict__ pmax,
                                                  const int* pred) {
  if (pred_off(pred)) return;
  const int s = blockIdx.y;
  const int h = (int)(plane / w);
  const double lim = sigma * thr[s];
  const int b = border ? border[s] : 0;
  const T* x = in + (size_t)s * plane;
  T* y = out + (size_t)s * plane;
  T m = -INFINITY;
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < plane; i += (size_t)gridDim.x * kT) {
    const T v = x[i];
    T o = ((double)fabs(v) > lim) ? v : (T)0;
    if (border) {
      const int r = (int)(i / w), c = (int)(i % w);
      if (r < b || r >= h - b || c < b || c >= w - b) o = 0;
    }
    y[i] = o;
    m = o > m ? o : m;
  }
  m = block_max_t<T>(m);
  if (threadIdx.x == 0) pmax[(size_t)s * gridDim.x + blockIdx.x] = m;
}

// per-plane max (or max |w|) of a plane stack: partials[s * gridDim.x + block]
template <class T>
__global__ __launch_bounds__(kT) void k_plane_max(const T* __restrict__ in, size_t plane, int use_abs,
                                                  T* __restrict__ pmax, const int* pred) {
  if (pred_off(pred)) return;
  const int s = blockIdx.y;
  const T* x = in + (size_t)s * plane;
  T m = -INFINITY;
  auto take = [&](T v) {
    const T a = use_abs ? (T)fabs(v) : v;
    m = a > m ? a : m;
  };
  const size_t stride = (size_t)gridDim.x * kT;
  size_t tail = 0;
  if constexpr (sizeof(T) == 4) {
    if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {  // float4 loads; the maximum does not depend on order
      const float4* x4 = reinterpret_cast<const float4*>(x);
      const size_t n4 = plane >> 2;
      for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < n4; i += stride) {
        const float4 a = x4[i];
        take(a.x), take(a.y), take(a.z), take(a.w);
      }
      tail = 4 * n4;
    }
  }
  for (size_t i = tail + blockIdx.x * (size_t)kT + threadIdx.x; i < plane; i += stride) take(x[i]);
  m = block_max_t<T>(m);
  if (threadIdx.x == 0) pmax[(size_t)s * gridDim.x + blockIdx.x] = m;
}

// per-plane reduce of partial maxima; out_max[s] (float) and optionally nsm[s] = max / energy[s]
// (one block per plane; max is exact in any order)
template <class T>
__global__ __launch_bounds__(kT) void k_max_final(const T* pmax, int nb, T* out_max, const double* energy,
                                                  double* nsm, const int* pred) {
  if (pred_off(pred)) return;
  const int s = blockIdx.x;
  T m = -INFINITY;
  for (int b = threadIdx.x; b < nb; b += kT) {
    const T v = pmax[(size_t)s * nb + b];
    m = v > m ? v : m;
  }
  m = block_max_t<T>(m);
  if (threadIdx.x == 0) {
    if (out_max) out_max[s] = m;
    if (nsm) nsm[s] = (double)m / energy[s];
  }
}

// ----------------------------------------------------------------------------- connected components
// A label word holds the index of the pixel's parent; in a root's own word the top bit is the keep
// rule's mark (planes hold fewer than 2^31 pixels).  Only set pixels have a label: which pixels are
// set is kept as one 64-bit word per row and 64 columns (layout (scale, row, word)), an eighth of a
// byte per pixel, so that every pass after the first reads 1/32 of the planes and touches labels and
// values of set pixels alone.
using u64 = unsigned long long;
constexpr int kMark = (int)0x80000000u;
constexpr int kCclW = 64, kCclH = 32;  // tile: one row is one wave's ballot

__host__ __device__ __forceinline__ int ccl_words(int wd) { return (wd + kCclW - 1) / kCclW; }
__host__ __device__ __forceinline__ int ccl_tiles(int h, int wd) { return ccl_words(wd) * ((h + kCclH - 1) / kCclH); }

__device__ __forceinline__ int ccl_find(const int* lab, int x) {
  int p = lab[x] & ~kMark;
  while (p != x) {
    x = p;
    p = lab[x] & ~kMark;
  }
  return x;
}

// before any mark is set
__device__ __forceinline__ void ccl_union(int* lab, int a, int b) {
  while (true) {
    a = ccl_find(lab, a);
    b = ccl_find(lab, b);
    if (a == b) return;
    if (a < b) {
      const int t = a;
      a = b;
      b = t;
    }
    const int old = atomicMin(&lab[a], b);
    if (old == a) return;
    a = old;
  }
}

__device__ __forceinline__ int lds_find(const int* L, int x) {
  int p = L[x];
  while (p != x) {
    x = p;
    p = L[x];
  }
  return x;
}

__device__ __forceinline__ void lds_union(int* L, int a, int b) {
  while (true) {
    a = lds_find(L, a);
    b = lds_find(L, b);
    if (a == b) return;
    if (a < b) {
      const int t = a;
      a = b;
      b = t;
    }
    const int old = atomicMin(&L[a], b);
    if (old == a) return;
    a = old;
  }
}

// Which unions with the row above a set pixel takes part in, given that its row neighbours are joined
// already: with the pixel above it, or the one above to the left, only where its run of set pixels
// starts (otherwise the pixel to the left has made that union), and with the one above to the right
// only where the pixel above is not set (otherwise both are one run).  m and u are the row's and the
// upper row's bits, the others those shifted by one pixel.
__device__ __forceinline__ void ccl_rules(u64 m, u64 left, u64 u, u64 ul, u64 ur, u64* up, u64* upl, u64* upr) {
  const u64 start = m & ~left;
  *up = start & u;
  *upl = start & ~u & ul;
  *upr = m & ~u & ur;
}

// this lane's bit of a mask that is the same in all lanes: the mask goes to the lanes' predicate as it is
__device__ __forceinline__ bool lane_bit(u64 mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }
__device__ __forceinline__ u64 first_lane(u64 v) {
  const unsigned lo = __builtin_amdgcn_readfirstlane((int)(unsigned)v);
  const unsigned hi = __builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32));
  return (u64)hi << 32 | lo;
}

// Two-level labelling, first level: one block labels a 64 x 32 tile in LDS (row runs linked to their
// first pixel by bit arithmetic on the row's ballot, then union-find with LDS atomicMin links between
// rows, so every tile component's root is its smallest raster index), and writes the rows' bit words
// and, for set pixels, the tile roots as global raster indices; a tile without a set pixel ends after
// the words.  The pass also takes the tile's maximum (of |w| with use_abs), so the planes are read
// once.  Bound: instruction issue and reading the planes in sparse tiles, the chains of dependent LDS
// reads in dense ones; a row is one wave's ballot, so the rows' words and union rules are scalar arithmetic; a
// wave unions its rows from the top down, which links each run straight to its component's root.
// NT threads (128 or 512) share a tile: four rows a wave end a tile soonest, sixteen spend the fewest
// instructions per pixel (source_extract_t chooses).  Seven 4096^2 planes take 144 / 161 / 241 us with
// 128 / 256 / 512 threads, five 500^2 planes 21.9 / 15.7 / 12.2 us.
template <class T, int NT>
__global__ __launch_bounds__(NT) void k_ccl_tile(const T* __restrict__ w, int* __restrict__ lab,
                                                    u64* __restrict__ bits, int h, int wd, int use_abs,
                                                    T* __restrict__ pmax, const int* pred) {
  if (pred_off(pred)) return;
  constexpr int TW = kCclW, TH = kCclH, PER = TH / (NT / 64);
  __shared__ int L[TH * TW];
  __shared__ u64 last_rows[NT / 64];  // each wave's last row
  const int s = blockIdx.y;
  const int nw = ccl_words(wd);
  const int cw = blockIdx.x % nw;
  const int r0 = (blockIdx.x / nw) * TH, c0 = cw * TW;
  const size_t plane = (size_t)h * wd;
  const T* x = w + (size_t)s * plane;
  int* l = lab + (size_t)s * plane;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = wave * PER;
  const int col = c0 + lane;
  const bool col_ok = col < wd;
  T v[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i)  // a lane or row outside the plane repeats a pixel of the tile
    v[i] = (x + (size_t)min(r0 + row0 + i, h - 1) * wd)[col_ok ? col : wd - 1];
  T m = -INFINITY;
  u64 word[PER];
  u64 any = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int r = r0 + row0 + i;
    const T a = use_abs ? (T)fabs(v[i]) : v[i];
    m = a > m ? a : m;
    word[i] = r < h ? __ballot(col_ok && v[i] != (T)0) : 0;
    any |= word[i];
    if (word[i] != 0) {
      const u64 gaps = ~word[i] & (((u64)1 << lane) - 1);
      if (lane_bit(word[i])) L[(row0 + i) * TW + lane] = (row0 + i) * TW + (gaps ? 64 - __clzll(gaps) : 0);
    }
  }
  // lane i stores row i's word
  u64 mine = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) mine = lane == i ? word[i] : mine;
  if (lane < PER && r0 + row0 + lane < h) bits[((size_t)s * h + r0 + row0 + lane) * nw + cw] = mine;
  if (lane == PER - 1) last_rows[wave] = mine;
  m = block_max_t<T>(m);
  if (threadIdx.x == 0) pmax[(size_t)s * gridDim.x + blockIdx.x] = m;
  if (!__syncthreads_or(any != 0)) return;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (word[i] == 0) continue;
    u64 u;
    if (i > 0)
      u = word[i > 0 ? i - 1 : 0];
    else
      u = wave > 0 ? first_lane(last_rows[wave > 0 ? wave - 1 : 0]) : 0;
    u64 up, upl, upr;
    ccl_rules(word[i], word[i] << 1, u, u << 1, u >> 1, &up, &upl, &upr);
    const int me = (row0 + i) * TW + lane;
    if (up && lane_bit(up)) lds_union(L, me, me - TW);
    if (upl && lane_bit(upl)) lds_union(L, me, me - TW - 1);
    if (upr && lane_bit(upr)) lds_union(L, me, me - TW + 1);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (word[i] == 0 || !lane_bit(word[i])) continue;
    const int root = lds_find(L, (row0 + i) * TW + lane);
    (l + (size_t)(r0 + row0 + i) * wd)[col] = (r0 + root / TW) * wd + c0 + root % TW;
  }
}

// Second level: unions across tile borders, so that pixels without a set neighbour across a border cost no label
// access.  On the rows that start a tile every pixel looks at the row above: a thread takes kCclPart pixels of a word
// there (a thread with a whole word makes up to 64 unions one after the other, each a chain of memory latencies: five
// 500 x 517 planes with 45% set pixels took 98 us, now 25).  On the others only the word's
// first and last pixel look at the neighbouring words, one thread a word, and not where the neighbour above or beside
// them makes the same union.  Unions commute: the roots, each component's smallest index, do not depend on
// their order.  The last block of a plane reduces the plane's tile maxima instead (smax).  Reading the labels of
// every tile border took 502 us on seven 4096^2 planes: with 32-pixel tiles that is every line of them.
constexpr int kCclPart = 4;
__host__ __device__ __forceinline__ unsigned ccl_border_items(int h, int wd) {  // words, then parts of the top rows' words
  return (unsigned)ccl_words(wd) * ((unsigned)h + (unsigned)((h + kCclH - 1) / kCclH) * (kCclW / kCclPart));
}
template <class T>
__global__ __launch_bounds__(kT) void k_ccl_border(int* __restrict__ lab, const u64* __restrict__ bits, int h, int wd,
                                                   const T* __restrict__ pmax, int n_pmax, T* __restrict__ smax,
                                                   const int* pred) {
  if (pred_off(pred)) return;
  const int s = blockIdx.y;
  if (blockIdx.x == gridDim.x - 1) {
    T m = -INFINITY;
    for (int i = threadIdx.x; i < n_pmax; i += kT) {
      const T v = pmax[(size_t)s * n_pmax + i];
      m = v > m ? v : m;
    }
    m = block_max_t<T>(m);
    if (threadIdx.x == 0) smax[s] = m;
    return;
  }
  const unsigned nw = ccl_words(wd);
  const unsigned n = (unsigned)h * nw, items = ccl_border_items(h, wd);
  int* l = lab + (size_t)s * h * wd;
  const u64* b = bits + (size_t)s * n;
  for (unsigned it = blockIdx.x * kT + threadIdx.x; it < items; it += (gridDim.x - 1) * kT) {
    const bool top = it >= n;
    unsigned i = it, part = 0;
    if (top) {
      const unsigned k = (it - n) / (kCclW / kCclPart);  // word k of the rows that start a tile
      part = (it - n) % (kCclW / kCclPart);
      i = k / nw * (kCclH * nw) + k % nw;
    }
    const u64 m = b[i];
    if (m == 0) continue;
    const int r = (int)(i / nw), cw = (int)(i - (unsigned)r * nw);
    if (!top && r % kCclH == 0) continue;
    const int me = r * wd + cw * kCclW;  // the word's first pixel
    const bool has_l = cw > 0, has_r = cw + 1 < (int)nw;
    const u64 lw = has_l ? b[i - 1] >> 63 : 0;  // the pixel left of the word
    const u64 u = r > 0 ? b[i - nw] : 0;
    const u64 ulw = r > 0 && has_l ? b[i - nw - 1] >> 63 : 0;
    const u64 urw = r > 0 && has_r ? b[i - nw + 1] & 1 : 0;
    if ((top ? part == 0 : !(u & ulw & 1)) && (lw & m & 1)) ccl_union(l, me, me - 1);
    if (top) {
      const u64 mine = (((u64)1 << kCclPart) - 1) << (part * kCclPart);
      u64 up, upl, upr;
      ccl_rules(m, (m << 1) | lw, u, (u << 1) | ulw, (u >> 1) | (urw << 63), &up, &upl, &upr);
      for (up &= mine; up; up &= up - 1) {
        const int c = me + __ffsll(up) - 1;
        ccl_union(l, c, c - wd);
      }
      for (upl &= mine; upl; upl &= upl - 1) {
        const int c = me + __ffsll(upl) - 1;
        ccl_union(l, c, c - wd - 1);
      }
      for (upr &= mine; upr; upr &= upr - 1) {
        const int c = me + __ffsll(upr) - 1;
        ccl_union(l, c, c - wd + 1);
      }
    } else {
      if (m & 1 & ulw & ~u & ~lw) ccl_union(l, me, me - wd - 1);
      if ((m >> 63) & urw & ~(u >> 63)) ccl_union(l, me + 63, me + 63 - wd + 1);
    }
  }
}

// labels for the caller: every set pixel's root without its mark, -1 for the others
__global__ __launch_bounds__(kT) void k_ccl_flatten(int* __restrict__ lab, const u64* __restrict__ bits, int h, int wd) {
  const int s = blockIdx.y;
  const size_t plane = (size_t)h * wd;
  const int nw = ccl_words(wd);
  int* l = lab + (size_t)s * plane;
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < plane; i += (size_t)gridDim.x * kT) {
    const int r = (int)(i / wd), c = (int)(i % wd);
    const bool on = (bits[((size_t)s * h + r) * nw + (c >> 6)] >> (c & 63)) & 1;
    l[i] = on ? ccl_find(l, (int)i) : -1;
  }
}

// Roots of the set ones (bits `on`) of four pixels from px on, walked side by side so that a step costs
// one memory latency for all of them; returns which of the roots carry the keep mark.  From the third link on a walk
// (HALVE) leaves each label pointing at its grandparent: the pixels of an object that winds through many tiles halve its
// chain of tile roots for one another (other walks read either link; roots, which carry the marks, are not written).
template <bool HALVE>
__device__ __forceinline__ unsigned ccl_find4(int* lab, int px, unsigned on, int (&root)[4]) {
  int child[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    root[k] = (on >> k) & 1 ? lab[px + k] & ~kMark : 0;
    child[k] = px + k;
  }
  unsigned marked = 0, more = on;
  for (int link = 1; more; ++link) {
    int p[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) p[k] = (more >> k) & 1 ? lab[root[k]] : 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (!((more >> k) & 1)) continue;
      if ((p[k] & ~kMark) == root[k]) {
        more &= ~(1u << k);
        marked |= p[k] < 0 ? 1u << k : 0u;
      } else if constexpr (HALVE) {
        if (link >= 3) lab[child[k]] = p[k];
        child[k] = root[k];
      }
      root[k] = p[k] & ~kMark;
    }
  }
  return marked;
}

// The first step of the keep rule of small stacks: links the set pixels of all scales (blockIdx.y) to their roots and
// marks the roots of the coarsest one's objects that hold a seed pixel (value >= tol * max).  A chain of tile roots is then
// walked here, for all scales at once, and not scale after scale in the steps that follow: the extraction on five 600^2
// planes of vertical lines takes 61 us (116 without this step), of one object winding through every tile 93 us (166).
template <class T>
__global__ __launch_bounds__(kT) void k_keep_first(const T* __restrict__ w, int* __restrict__ lab,
                                                   const u64* __restrict__ bits, int S, const T* __restrict__ smax,
                                                   double tol, int neg_comp, int h, int wd, const int* pred) {
  if (pred_off(pred)) return;
  const int s = blockIdx.y;
  const unsigned nq = (unsigned)(wd + 3) / 4;
  const unsigned i = blockIdx.x * (unsigned)kT + threadIdx.x;
  if (i >= (unsigned)h * nq) return;
  const int r = (int)(i / nq), c = 4 * (int)(i - (unsigned)r * nq);
  const unsigned on = (unsigned)(bits[((size_t)s * h + r) * ccl_words(wd) + (c >> 6)] >> (c & 63)) & 15u;
  if (on == 0) return;
  const size_t o = (size_t)s * h * wd;
  const int px = r * wd + c;
  int* l = lab + o;
  const bool mark = s == S - 1;
  T v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = mark && ((on >> k) & 1) ? w[o + px + k] : (T)0;
  const double lim = mark ? tol * (double)smax[s] : 0.0;
  int root[4];
  (void)ccl_find4<true>(l, px, on, root);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (!((on >> k) & 1)) continue;
    if (root[k] != px + k && l[px + k] != root[k]) l[px + k] = root[k];  // a root's own word is left: it takes the mark
    if (mark && (double)(neg_comp ? (T)fabs(v[k]) : v[k]) >= lim) l[root[k]] = root[k] | kMark;
  }
}

// One step of the per-scale keep rule, coarsest scale first, in one pass over the pixels: applies
// scale sa's marks (mask = pixel's object kept, extracted = mask * w) and marks the roots of scale
// sm = sa - 1's objects that hold a seed pixel (value >= tol * max) inside sa's kept mask.  sa < 0:
// mark only (the coarsest scale, which has no coarser mask); sm < 0: apply only.  A thread takes U times four
// pixels of a row: their bits come from the scales' words, requested for all of them first, labels
// and values are read at set pixels
// alone, and VEC (sides and buffers that keep quads aligned) writes the four extracted values and the
// four mask bytes as one store each, with U > 1 past the caches: the extraction of seven 4096^2 planes takes 477 us
// (499 through them), of three 3000^2 planes 115 us (139), which a reader of the outputs pays back only there (191
// and 190 us with one).  Roots are found by walking from the tile's root, so on large stacks no pass
// compresses the labels beforehand (162 us on seven 4096^2 planes; k_keep_first does on small ones).  Bound: the two
// outputs' stores: 31 us a scale at 4096^2 (64 us on label planes with separate flags; 33 us with one quad a thread).
template <class T, bool VEC, int U>
__global__ __launch_bounds__(kT) void k_keep_step(const T* __restrict__ w, int* __restrict__ lab,
                                                  const u64* __restrict__ bits, int sa, int sm,
                                                  const T* __restrict__ smax, double tol, int neg_comp, int h, int wd,
                                                  uint8_t* __restrict__ mask, T* __restrict__ extracted,
                                                  const int* pred) {
  if (pred_off(pred)) return;
  const int nw = ccl_words(wd);
  const unsigned nq = (unsigned)(wd + 3) / 4;
  const size_t plane = (size_t)h * wd;
  const size_t oa = (size_t)(sa < 0 ? 0 : sa) * plane, om = (size_t)(sm < 0 ? 0 : sm) * plane;
  int* la = lab + oa;
  int* lm = lab + om;
  const u64* ba = bits + (size_t)(sa < 0 ? 0 : sa) * h * nw;
  const u64* bm = bits + (size_t)(sm < 0 ? 0 : sm) * h * nw;
  const unsigned total = (unsigned)h * nq;
  const unsigned i0 = blockIdx.x * (unsigned)(kT * U) + threadIdx.x;
  int px[U], c[U];
  unsigned on_a[U], on_m[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const unsigned i = min(i0 + u * kT, total - 1);
    const int r = (int)(i / nq);
    c[u] = 4 * (int)(i - (unsigned)r * nq);
    px[u] = r * wd + c[u];
    const int word = r * nw + (c[u] >> 6), shift = c[u] & 63;
    on_a[u] = (unsigned)(ba[word] >> shift) & 15u;
    on_m[u] = (unsigned)(bm[word] >> shift) & 15u;
  }
  const double lim = sm >= 0 ? tol * (double)smax[sm] : 0.0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (i0 + u * kT >= total) return;
    unsigned kept = 15u;
    int root[4];
    if (sa >= 0) {
      const unsigned on = on_a[u];
      Quad<T> e;
#pragma unroll
      for (int k = 0; k < 4; ++k) e.a[k] = (on >> k) & 1 ? w[oa + px[u] + k] : (T)0;
      kept = on ? ccl_find4<U == 1>(la, px[u], on, root) : 0u;
#pragma unroll
      for (int k = 0; k < 4; ++k) e.a[k] = (kept >> k) & 1 ? e.a[k] : (T)0;
      uint8_t* mo = mask + oa + px[u];
      T* eo = extracted ? extracted + oa + px[u] : nullptr;
      if constexpr (VEC) {
        const uint32_t m4 = (kept & 1u) | ((kept & 2u) << 7) | ((kept & 4u) << 14) | ((kept & 8u) << 21);
        if constexpr (U > 1) {
          __builtin_nontemporal_store(m4, reinterpret_cast<uint32_t*>(mo));
          if (eo) store_stream(eo, e);
        } else {
          *reinterpret_cast<uint32_t*>(mo) = m4;
          if (eo) *reinterpret_cast<Quad<T>*>(eo) = e;
        }
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (c[u] + k >= wd) break;
          mo[k] = (kept >> k) & 1u;
          if (eo) eo[k] = e.a[k];
        }
      }
    }
    if (sm < 0) continue;
    unsigned seeds = on_m[u] & kept;
    if (!seeds) continue;
    T x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] = (seeds >> k) & 1 ? w[om + px[u] + k] : (T)0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const T v = neg_comp ? (T)fabs(x[k]) : x[k];
      if (!((double)v >= lim)) seeds &= ~(1u << k);
    }
    if (!seeds) continue;
    (void)ccl_find4<U == 1>(lm, px[u], seeds, root);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if ((seeds >> k) & 1) lm[root[k]] = root[k] | kMark;
  }
}

// raster-order label numbering: count roots per block, scan, write ranks
__global__ __launch_bounds__(kT) void k_root_count(const int* __restrict__ lab, size_t plane, int chunk,
                                                   uint32_t* __restrict__ counts) {
  const int s = blockIdx.y;
  const int* l = lab + (size_t)s * plane;
  const size_t lo = (size_t)blockIdx.x * chunk;
  const size_t hi = min(plane, lo + (size_t)chunk);
  uint32_t c = 0;
  for (size_t i = lo + threadIdx.x; i < hi; i += kT) c += (l[i] == (int)i);
  __shared__ uint32_t red[kT];
  red[threadIdx.x] = c;
  __syncthreads();
  for (int o = kT / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) counts[(size_t)s * gridDim.x + blockIdx.x] = red[0];
}

__global__ void k_root_scan(uint32_t* counts, int nb, int S, uint32_t* totals) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  uint32_t run = 0;
  for (int b = 0; b < nb; ++b) {
    const uint32_t v = counts[(size_t)s * nb + b];
    counts[(size_t)s * nb + b] = run;
    run += v;
  }
  if (totals) totals[s] = run;
}

// serial-in-chunk ranks (one thread per chunk keeps raster order), then label each pixel by its root's rank
__global__ void k_root_rank(int* __restrict__ lab, size_t plane, int chunk, const uint32_t* __restrict__ offs,
                            int nb, int* __restrict__ rank) {
  const int s = blockIdx.y;
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  const int* l = lab + (size_t)s * plane;
  int* rk = rank + (size_t)s * plane;
  uint32_t run = offs[(size_t)s * nb + b];
  const size_t lo = (size_t)b * chunk;
  const size_t hi = min(plane, lo + (size_t)chunk);
  for (size_t i = lo; i < hi; ++i)
    if (l[i] == (int)i) rk[i] = (int)(++run);
}

__global__ __launch_bounds__(kT) void k_label_out(const int* __restrict__ lab, const int* __restrict__ rank,
                                                  size_t plane, int* __restrict__ out) {
  const int s = blockIdx.y;
  const int* l = lab + (size_t)s * plane;
  const int* rk = rank + (size_t)s * plane;
  int* o = out + (size_t)s * plane;
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < plane; i += (size_t)gridDim.x * kT)
    o[i] = (l[i] >= 0) ? rk[l[i]] : 0;
}

// ----------------------------------------------------------------------------- reductions & CG vectors
// partial[b] = sum over the block's grid-stride range of a[i]*b[i] (b == null: a[i]^2)
template <class T>
__global__ __launch_bounds__(kT) void k_dot(const T* __restrict__ a, const T* __restrict__ b, size_t n,
                                            double* __restrict__ partial, const int* pred) {
  if (pred_off(pred)) return;
  double acc = 0.0;
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < n; i += (size_t)gridDim.x * kT) {
    const double x = a[i];
    acc = fma(x, b ? (double)b[i] : x, acc);
  }
  acc = block_sum_f64(acc);
  if (threadIdx.x == 0) partial[blockIdx.x] = acc;
}

// per-plane sums of squares of a plane stack: partial[s * gridDim.x + block]
template <class T>
__global__ __launch_bounds__(kT) void k_plane_sumsq(const T* __restrict__ a, size_t plane,
                                                    double* __restrict__ partial, const int* pred) {
  if (pred_off(pred)) return;
  const int s = blockIdx.y;
  const T* x = a + (size_t)s * plane;
  double acc = 0.0;
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < plane; i += (size_t)gridDim.x * kT) {
    const double v = x[i];
    acc = fma(v, v, acc);
  }
  acc = block_sum_f64(acc);
  if (threadIdx.x == 0) partial[(size_t)s * gridDim.x + blockIdx.x] = acc;
}

// sum of (x - mean)^2 where mean = *mean_sum / count
template <class T>
__global__ __launch_bounds__(kT) void k_dev2(const T* __restrict__ a, size_t n, const double* __restrict__ sum,
                                             double* __restrict__ partial) {
  const double mean = *sum / (double)n;
  double acc = 0.0;
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < n; i += (size_t)gridDim.x * kT) {
    const double d = (double)a[i] - mean;
    acc = fma(d, d, acc);
  }
  acc = block_sum_f64(acc);
  if (threadIdx.x == 0) partial[blockIdx.x] = acc;
}

template <class T>
__global__ __launch_bounds__(kT) void k_sum(const T* __restrict__ a, size_t n, double* __restrict__ partial) {
  double acc = 0.0;
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < n; i += (size_t)gridDim.x * kT) acc += (double)a[i];
  acc = block_sum_f64(acc);
  if (threadIdx.x == 0) partial[blockIdx.x] = acc;
}

// out[g] = sum of partial[g*np .. g*np + np) in a fixed order (one block per group)
__global__ __launch_bounds__(kT) void k_sum_partials(const double* __restrict__ partial, long np,
                                                     double* __restrict__ out, const int* pred) {
  if (pred_off(pred)) return;
  const double* p = partial + (size_t)blockIdx.x * np;
  double acc = 0.0;
  for (long i = threadIdx.x; i < np; i += kT) acc += p[i];
  acc = block_sum_f64(acc);
  if (threadIdx.x == 0) out[blockIdx.x] = acc;
}

struct SumBatch {
  const double* partial[kMaxBatch];
  long np[kMaxBatch];
  double* out[kMaxBatch];
  const int* pred[kMaxBatch];
};

// job blockIdx.x: same summation order as k_sum_partials for one group
__global__ __launch_bounds__(kT) void k_sum_partials_batch(SumBatch b) {
  if (pred_off(b.pred[blockIdx.x])) return;
  const double* p = b.partial[blockIdx.x];
  const long np = b.np[blockIdx.x];
  double acc = 0.0;
  for (long i = threadIdx.x; i < np; i += kT) acc += p[i];
  acc = block_sum_f64(acc);
  if (threadIdx.x == 0) *b.out[blockIdx.x] = acc;
}

}  // namespace

// ============================================================================= host wrappers
static int ew_grid(size_t n) {
  size_t b = (n + (size_t)kT * 4 - 1) / ((size_t)kT * 4);
  if (b < 1) b = 1;
  if (b > 2048) b = 2048;
  return (int)b;
}

int reduce_grid(size_t n) { return ew_grid(n); }

static bool aligned16(const void* a, const void* b = nullptr) {
  return ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15) == 0;
}

// Whether an output of this many bytes is stored past the caches: one that does not fit the last-level cache (256 MB)
// is gone from it before it is read again, and evicts what the launch itself reads.
static bool past_caches(size_t bytes) { return bytes > (size_t)256 << 20; }

// blocks for a 16-byte streaming kernel doing four accesses per thread
static int vec_grid(size_t n) {
  size_t b = ((n >> 2) + (size_t)kT * 4 - 1) / ((size_t)kT * 4);
  if (b < 1) b = 1;
  if (b > 16384) b = 16384;
  return (int)b;
}

void copy_plane(const float* src, float* dst, size_t n, const int* pred, hipStream_t st) {
  if (aligned16(src, dst))
    hipLaunchKernelGGL(k_copy, dim3(vec_grid(n)), dim3(kT), 0, st, src, dst, n, pred);
  else
    hipLaunchKernelGGL(k_copy1<float>, dim3(ew_grid(n)), dim3(kT), 0, st, src, dst, n, pred);
  PMS_LAUNCH_CHECK();
}

// a double plane is copied as twice as many floats (bit copy)
void copy_plane(const double* src, double* dst, size_t n, const int* pred, hipStream_t st) {
  copy_plane(reinterpret_cast<const float*>(src), reinterpret_cast<float*>(dst), 2 * n, pred, st);
}

template <class T>
static void masked_copy_t(const T* src, const uint8_t* mask, T* dst, size_t n, const int* pred, hipStream_t st) {
  hipLaunchKernelGGL(k_masked_copy<T>, dim3(ew_grid(n)), dim3(kT), 0, st, src, mask, dst, n, pred);
  PMS_LAUNCH_CHECK();
}
void masked_copy(const float* src, const uint8_t* mask, float* dst, size_t n, const int* pred, hipStream_t st) {
  masked_copy_t(src, mask, dst, n, pred, st);
}
void masked_copy(const double* src, const uint8_t* mask, double* dst, size_t n, const int* pred, hipStream_t st) {
  masked_copy_t(src, mask, dst, n, pred, st);
}

void fill_f32(float* p, size_t n, float v, hipStream_t st) {
  if (aligned16(p))
    hipLaunchKernelGGL(k_fill16<float>, dim3(vec_grid(n)), dim3(kT), 0, st, p, n, v);
  else
    hipLaunchKernelGGL(k_fill_f32, dim3(ew_grid(n)), dim3(kT), 0, st, p, n, v);
  PMS_LAUNCH_CHECK();
}

void fill_u32(uint32_t* p, size_t n, uint32_t v, hipStream_t st) {
  if (aligned16(p))
    hipLaunchKernelGGL(k_fill16<uint32_t>, dim3(vec_grid(n)), dim3(kT), 0, st, p, n, v);
  else
    hipLaunchKernelGGL(k_fill_u32, dim3(ew_grid(n)), dim3(kT), 0, st, p, n, v);
  PMS_LAUNCH_CHECK();
}

void fill_zero(float* p, size_t n, hipStream_t st) { fill_u32(reinterpret_cast<uint32_t*>(p), n, 0u, st); }
void fill_zero(double* p, size_t n, hipStream_t st) { fill_u32(reinterpret_cast<uint32_t*>(p), 2 * n, 0u, st); }

template <class T, class TIN>
static void window_copy_t(const TIN* src, int ld, int r0, int c0, int n, const T* mul, T* dst, hipStream_t st) {
  hipLaunchKernelGGL((k_window<T, TIN>), dim3(ew_grid((size_t)n * n)), dim3(kT), 0, st, src, ld, r0, c0, n, mul,
                     dst);
  PMS_LAUNCH_CHECK();
}
void window_copy(const float* src, int ld, int r0, int c0, int n, const float* mul, float* dst, hipStream_t st) {
  window_copy_t(src, ld, r0, c0, n, mul, dst, st);
}
void window_copy(const float* src, int ld, int r0, int c0, int n, const double* mul, double* dst, hipStream_t st) {
  window_copy_t(src, ld, r0, c0, n, mul, dst, st);
}
void window_copy(const double* src, int ld, int r0, int c0, int n, const double* mul, double* dst, hipStream_t st) {
  window_copy_t(src, ld, r0, c0, n, mul, dst, st);
}

// Python slice(start, stop).indices(n) for step 1, as [lo, hi) with hi >= lo
static void py_slice(long start, long stop, long n, int* lo, int* hi) {
  auto fix = [n](long v) {
    if (v < 0) v += n;
    if (v < 0) v = 0;
    if (v > n) v = n;
    return v;
  };
  long a = fix(start), b = fix(stop);
  if (b < a) b = a;
  *lo = (int)a;
  *hi = (int)b;
}

NoiseMask noise_mask(int h, int w, int edge_excl, int int_excl) {
  NoiseMask m{};
  m.masked = (edge_excl != 0) || (int_excl != 0);
  m.inc_r0 = 0;
  m.inc_r1 = h;
  m.inc_c0 = 0;
  m.inc_c1 = w;
  m.exc_r0 = m.exc_r1 = m.exc_c0 = m.exc_c1 = 0;
  if (edge_excl != 0) {
    py_slice(edge_excl, -edge_excl, h, &m.inc_r0, &m.inc_r1);
    py_slice(edge_excl, -edge_excl, w, &m.inc_c0, &m.inc_c1);
  }
  if (int_excl != 0) {
    // iuwt_toolbox.py:29,40: mid = in1.shape[1]/2 is the row count of the (scales, rows, cols) stack,
    // and the same mid bounds both axes
    const int mid = h / 2;
    py_slice(mid - int_excl, mid + int_excl, h, &m.exc_r0, &m.exc_r1);
    py_slice(mid - int_excl, mid + int_excl, w, &m.exc_c0, &m.exc_c1);
  }
  const long inc = (long)(m.inc_r1 - m.inc_r0) * (m.inc_c1 - m.inc_c0);
  const int ir0 = std::max(m.inc_r0, m.exc_r0), ir1 = std::min(m.inc_r1, m.exc_r1);
  const int ic0 = std::max(m.inc_c0, m.exc_c0), ic1 = std::min(m.inc_c1, m.exc_c1);
  const long ov = (ir1 > ir0 && ic1 > ic0) ? (long)(ir1 - ir0) * (ic1 - ic0) : 0;
  m.count = inc - ov;
  return m;
}

// workspace layout: [ranges: 16 slots][bins: 16 x kMadBins][keys set aside: S planes of mad_room keys]
// [keys of the median's bin: S planes of mad_list_room keys].  Nothing in it has to be prepared.
static size_t mad_aside_offset() { return (size_t)kMaxPlanes * (kRangeBytes + kMadBins * sizeof(uint32_t)); }
size_t mad_work_bytes(int S, size_t plane, size_t real_bytes) {
  return mad_aside_offset() + (size_t)S * (mad_room(plane) + mad_list_room(plane)) * real_bytes;
}

// Allocation-free median workspace: one file-scope device array per GPU, holding the select state
// and histograms of one call of up to kMaxPlanes planes (131,584 bytes).  Host code never names
// the array in a kernel argument or copy: the array's host-side symbol is a stand-in, not a
// device address, so each device's address is looked up once with hipGetSymbolAddress (with that
// device current) and kept here.
namespace {
constexpr size_t kNoAllocMadBytes = (size_t)kMaxPlanes * (kSelBytes + kBins * sizeof(uint32_t));
static __device__ __align__(256) unsigned char scratch[kNoAllocMadBytes];
std::mutex g_scratch_mu;
std::map<int, void*> g_scratch_ptr;
}  // namespace

size_t noalloc_mad_bytes() { return kNoAllocMadBytes; }

void* noalloc_mad_scratch() {
  int dev = 0;
  PMS_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  auto it = g_scratch_ptr.find(dev);
  if (it != g_scratch_ptr.end()) return it->second;
  void* ptr = nullptr;
  PMS_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  PMS_REQUIRE(ptr != nullptr, "device scratch symbol has no address");
  g_scratch_ptr.emplace(dev, ptr);
  return ptr;
}

static void mad_select_init(void* work, hipStream_t st) {
  uint32_t* hist = (uint32_t*)((char*)work + (size_t)kMaxPlanes * kSelBytes);
  fill_u32(hist, (size_t)kMaxPlanes * kBins, 0u, st);
}

static void check_mad(int S, const NoiseMask& nm) {
  PMS_REQUIRE(nm.count > 0, "noise mask selects no pixels");
  PMS_REQUIRE(nm.count < (1L << 32), "plane too large for the median");
  PMS_REQUIRE(S >= 1 && S <= kMaxPlanes, "the median handles 1..16 planes per call");
}

// Exact median per plane for a workspace of kNoAllocMadBytes: radix select over the key bits in digits of at most
// 11 bits (11/11/10), one histogram pass and one select step per digit; for even counts the last pass and select
// also find the successor of the low median.
void mad_thresholds_noalloc(const float* planes, int S, int h, int w, const NoiseMask& nm, double* thr, void* work,
                            const int* pred, hipStream_t st) {
  check_mad(S, nm);
  // the histograms hold the previous call's contents (the select state is rewritten by the first kernel)
  mad_select_init(work, st);
  SelState* sst = (SelState*)work;
  uint32_t* hist = (uint32_t*)((char*)work + (size_t)kMaxPlanes * kSelBytes);
  const size_t plane = (size_t)h * w;
  Rect inc{nm.inc_r0, nm.inc_r1, nm.inc_c0, nm.inc_c1};
  Rect exc{nm.exc_r0, nm.exc_r1, nm.exc_c0, nm.exc_c1};
  hipLaunchKernelGGL(k_mad_init, dim3(ceil_div(S, 64)), dim3(64), 0, st, sst, S, (uint32_t)nm.count);
  PMS_LAUNCH_CHECK();
  const int gx = std::min(ew_grid(plane), 512);
  constexpr int shifts[] = {21, 10, 0}, bits[] = {11, 11, 10};
  const int above = (nm.count & 1) == 0 ? 1 : 0;
  for (int pass = 0; pass < 3; ++pass) {
    const int pshift = pass == 0 ? 32 : shifts[pass - 1], ab = pass == 2 ? above : 0;
    hipLaunchKernelGGL((nm.masked ? k_mad_hist<true> : k_mad_hist<false>), dim3(gx, S), dim3(kT), 0, st, planes, plane, w,
                       inc, exc, shifts[pass], bits[pass], pshift, ab, sst, hist, pred);
    PMS_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_mad_select, dim3(S), dim3(kT), 0, st, sst, hist, shifts[pass], bits[pass], pass == 2, pred);
    PMS_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_mad_finish, dim3(ceil_div(S, 64)), dim3(64), 0, st, (const SelState*)sst, S, thr, pred);
  PMS_LAUNCH_CHECK();
}

// Exact median per plane in one reading of it (k_mad_one, or k_mad_pivot / k_mad_scan / k_mad_pick).
// The sample has 8192 keys below 2^20 noise pixels and 16384 above: a range of 8.8 and 6.3% of the
// plane (32768: 4.4%, 35 instead of 20 us in k_mad_pivot for 4 us less in k_mad_scan).  From 2^20 pixels on the
// median's bin is collected by many blocks: one block alone needs 45 us to look at what a 4096^2 plane sets
// aside.  Seven 4096^2 planes take 160 us (285 us with the radix select), five 500^2 planes with an edge
// mask 37 us (50 us), four 256^2 planes 26 us (33 us).  Seven planes with many equal keys (48 to 52% zeros, two values, 30
// whole numbers, values within 1e-5 of one) take 132 to 260 us (277 to 810 us with the radix select; 1.1 to 22 ms with the
// ends in the range and one block selecting from the plane), float64 ones 260 to 450 us (1.2 to 1.4 ms; 2.1 to 47 ms).
template <class T, bool MASKED>
static void mad_thresholds_t(const T* planes, int S, int h, int w, const NoiseMask& nm, double* thr, void* work,
                             const int* pred, hipStream_t st) {
  using K = typename MadKey<T>::K;
  check_mad(S, nm);
  const size_t plane = (size_t)h * w;
  const Rect inc{nm.inc_r0, nm.inc_r1, nm.inc_c0, nm.inc_c1};
  const Rect exc{nm.exc_r0, nm.exc_r1, nm.exc_c0, nm.exc_c1};
  const size_t area = (size_t)(inc.r1 - inc.r0) * (inc.c1 - inc.c0);
  const uint32_t n = (uint32_t)nm.count;
  if constexpr (sizeof(T) == 4) {
    // 32-bit pixel numbers end here; the counts are of the pixels left in, which check_mad bounds
    if (area >= (size_t)1 << 32) return mad_thresholds_noalloc(planes, S, h, w, nm, thr, work, pred, st);
  }
  PMS_REQUIRE(area < ((size_t)1 << 32), "plane too large for the median");
  if (area <= (size_t)kMadOne) {
    auto one = area <= (size_t)8 * kMT ? k_mad_one<T, MASKED, 8> : k_mad_one<T, MASKED, 32>;
    hipLaunchKernelGGL(one, dim3(S), dim3(kMT), 0, st, planes, plane, w, inc, exc, (uint32_t)area, n, thr, pred);
    PMS_LAUNCH_CHECK();
    return;
  }
  MadRange<K>* range = (MadRange<K>*)work;
  uint32_t* hist = (uint32_t*)((char*)work + (size_t)kMaxPlanes * kRangeBytes);
  const size_t room = mad_room(plane), list_room = mad_list_room(plane);
  K* aside = (K*)((char*)work + mad_aside_offset());
  K* lists = aside + (size_t)S * room;
  const bool large = area >= (size_t)1 << 20;
  auto pivot = large ? k_mad_pivot<T, MASKED, 16> : k_mad_pivot<T, MASKED, 8>;
  hipLaunchKernelGGL(pivot, dim3(S), dim3(kMT), 0, st, planes, plane, w, inc, exc, (uint32_t)area, range, hist, pred);
  PMS_LAUNCH_CHECK();
  // one group of keys a thread until 512 blocks a plane
  const int gx = (int)std::min<size_t>((area + kT * (32 / sizeof(T)) - 1) / (kT * (32 / sizeof(T))), 512);
  hipLaunchKernelGGL((k_mad_scan<T, MASKED>), dim3(gx, S), dim3(kT), 0, st, planes, plane, w, inc, exc, range, hist,
                     aside, room, pred);
  PMS_LAUNCH_CHECK();
  if (large) {
    hipLaunchKernelGGL((k_mad_collect<T>), dim3(32, S), dim3(kMT), 0, st, n, range, (const uint32_t*)hist,
                       (const K*)aside, room, lists, list_room, pred);
    PMS_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL((k_mad_pick<T, MASKED>), dim3(S), dim3(kMT), 0, st, planes, plane, w, inc, exc, n,
                     (const MadRange<K>*)range, (const uint32_t*)hist, (const K*)aside, room,
                     large ? (const K*)lists : (const K*)nullptr, list_room, thr, pred);
  PMS_LAUNCH_CHECK();
}
template <class T>
static void mad_thresholds_any(const T* planes, int S, int h, int w, const NoiseMask& nm, double* thr, void* work,
                               const int* pred, hipStream_t st) {
  if (nm.masked)
    mad_thresholds_t<T, true>(planes, S, h, w, nm, thr, work, pred, st);
  else
    mad_thresholds_t<T, false>(planes, S, h, w, nm, thr, work, pred, st);
}
void mad_thresholds(const float* planes, int S, int h, int w, const NoiseMask& nm, double* thr, void* work,
                    const int* pred, hipStream_t st) {
  mad_thresholds_any(planes, S, h, w, nm, thr, work, pred, st);
}
void mad_thresholds(const double* planes, int S, int h, int w, const NoiseMask& nm, double* thr, void* work,
                    const int* pred, hipStream_t st) {
  mad_thresholds_any(planes, S, h, w, nm, thr, work, pred, st);
}

int threshold_grid(size_t plane) { return std::min(ew_grid(plane), 256); }

template <class T>
static void apply_threshold_t(const T* in, T* out, int S, int h, int w, const double* thr, double sigma,
                              const int* border, T* pmax, const int* pred, hipStream_t st) {
  const size_t plane = (size_t)h * w;
  const int gx = threshold_grid(plane);
  const bool vec = plane % 4 == 0 && aligned16(in, out) && (!border || w % 4 == 0);
  const bool stream = past_caches(plane * S * sizeof(T));
  hipLaunchKernelGGL((!vec ? k_threshold<T> : stream ? k_threshold4<T, true> : k_threshold4<T, false>), dim3(gx, S), dim3(kT),
                     0, st, in, out, plane, w, thr, sigma, border, pmax, pred);
  PMS_LAUNCH_CHECK();
}
void apply_threshold(const float* in, float* out, int S, int h, int w, const double* thr, double sigma,
                     const int* border, float* pmax, const int* pred, hipStream_t st) {
  apply_threshold_t(in, out, S, h, w, thr, sigma, border, pmax, pred, st);
}
void apply_threshold(const double* in, double* out, int S, int h, int w, const double* thr, double sigma,
                     const int* border, double* pmax, const int* pred, hipStream_t st) {
  apply_threshold_t(in, out, S, h, w, thr, sigma, border, pmax, pred, st);
}

template <class T>
static void plane_max_t(const T* in, int S, size_t plane, int use_abs, T* pmax, const int* pred, hipStream_t st) {
  const int gx = threshold_grid(plane);
  hipLaunchKernelGGL(k_plane_max<T>, dim3(gx, S), dim3(kT), 0, st, in, plane, use_abs, pmax, pred);
  PMS_LAUNCH_CHECK();
}
void plane_max(const float* in, int S, size_t plane, int use_abs, float* pmax, const int* pred, hipStream_t st) {
  plane_max_t(in, S, plane, use_abs, pmax, pred, st);
}
void plane_max(const double* in, int S, size_t plane, int use_abs, double* pmax, const int* pred, hipStream_t st) {
  plane_max_t(in, S, plane, use_abs, pmax, pred, st);
}

template <class T>
static void max_final_t(const T* pmax, int nb, int S, T* out_max, const double* energy, double* nsm, const int* pred,
                        hipStream_t st) {
  hipLaunchKernelGGL(k_max_final<T>, dim3(S), dim3(kT), 0, st, pmax, nb, out_max, energy, nsm, pred);
  PMS_LAUNCH_CHECK();
}
void max_final(const float* pmax, int nb, int S, float* out_max, const double* energy, double* nsm, const int* pred,
               hipStream_t st) {
  max_final_t(pmax, nb, S, out_max, energy, nsm, pred, st);
}
void max_final(const double* pmax, int nb, int S, double* out_max, const double* energy, double* nsm,
               const int* pred, hipStream_t st) {
  max_final_t(pmax, nb, S, out_max, energy, nsm, pred, st);
}

// workspace layout: [maxima: 64 values][tile maxima: S x tiles values][set-pixel words: S x h x words]
// [labels: S planes of int], values sized for double so that one layout serves both element types.
// Nothing in it has to be prepared: every part is written before it is read.
static size_t ext_round(size_t bytes) { return ((bytes + 255) / 256) * 256; }
static size_t ext_bits_offset(int S, int h, int wd) {
  return ext_round((64 + (size_t)S * ccl_tiles(h, wd)) * sizeof(double));
}
static size_t ext_labels_offset(int S, int h, int wd) {
  return ext_bits_offset(S, h, wd) + ext_round((size_t)S * h * ccl_words(wd) * sizeof(u64));
}

// The words and tiles of a plane and of its transpose differ in number: room for either, as one workspace may serve both.
size_t extract_work_bytes(int S, int h, int w) {
  return std::max(ext_labels_offset(S, h, w), ext_labels_offset(S, w, h)) + (size_t)S * h * w * sizeof(int);
}

template <class T>
static void source_extract_t(const T* w, int S, int h, int wd, double tol, int neg_comp, uint8_t* mask, T* extracted,
                             int* labels_out, void* work, const int* pred, hipStream_t st) {
  PMS_REQUIRE((size_t)h * wd < (size_t)1 << 31, "plane too large for int labels");
  PMS_REQUIRE(S >= 1 && S <= kMaxPlanes, "source extraction handles 1..16 planes per call");
  const size_t plane = (size_t)h * wd;
  T* smax = (T*)work;
  T* pmax = (T*)((char*)work + 64 * sizeof(double));
  u64* bits = (u64*)((char*)work + ext_bits_offset(S, h, wd));
  int* lab = (int*)((char*)work + ext_labels_offset(S, h, wd));
  const int tiles = ccl_tiles(h, wd);
  // While every tile's block is resident at once (1024 blocks of 512 threads), the time is that of one
  // tile; beyond, it is the instructions of all.
  if ((size_t)tiles * S <= 1024)
    hipLaunchKernelGGL((k_ccl_tile<T, 512>), dim3(tiles, S), dim3(512), 0, st, w, lab, bits, h, wd, neg_comp, pmax,
                       pred);
  else
    hipLaunchKernelGGL((k_ccl_tile<T, 128>), dim3(tiles, S), dim3(128), 0, st, w, lab, bits, h, wd, neg_comp, pmax,
                       pred);
  PMS_LAUNCH_CHECK();
  const int gb = (int)std::min<unsigned>((ccl_border_items(h, wd) + kT - 1) / kT, 1024);
  hipLaunchKernelGGL(k_ccl_border<T>, dim3(gb + 1, S), dim3(kT), 0, st, lab, (const u64*)bits, h, wd, (const T*)pmax,
                     tiles, smax, pred);
  PMS_LAUNCH_CHECK();
  // keep rule from the coarsest scale down: mark S-1; apply s and mark s-1; ...; apply 0
  const bool vec = wd % 4 == 0 && aligned16(extracted) && (reinterpret_cast<uintptr_t>(mask) & 3) == 0;
  const unsigned quads = (unsigned)h * (unsigned)ceil_div(wd, 4);
  // four quads a thread once that still leaves eight blocks per CU (from about 2900^2 pixels on);
  // below, a thread's chain of dependent reads sets the time and more threads hide it
  const bool four = quads >= 4u * kT * 2048;
  const unsigned per = kT * (four ? 4 : 1);
  auto keep = vec ? (four ? k_keep_step<T, true, 4> : k_keep_step<T, true, 1>)
                  : (four ? k_keep_step<T, false, 4> : k_keep_step<T, false, 1>);
  // On more tiles the walks of a step's pixels hide behind one another, and reading every label once more costs more than it
  // saves: 1% set pixels on five 600^2 planes (950 tiles) 34 -> 32 us, on seven of 700^2 (1694) 46 -> 49, three of 1400^2
  // (2904) 39 -> 44; lines and winding objects there 162 -> 95, 338 -> 153 and 152 -> 105, 191 -> 139.
  const bool first = (size_t)tiles * S <= 2048;
  if (first) {
    hipLaunchKernelGGL(k_keep_first<T>, dim3((quads + kT - 1) / kT, S), dim3(kT), 0, st, w, lab, (const u64*)bits, S,
                       (const T*)smax, tol, neg_comp, h, wd, pred);
    PMS_LAUNCH_CHECK();
  }
  for (int sa = first ? S - 1 : S; sa >= 0; --sa) {
    hipLaunchKernelGGL(keep, dim3((quads + per - 1) / per), dim3(kT), 0, st, w, lab, (const u64*)bits,
                       sa < S ? sa : -1, sa - 1, (const T*)smax, tol, neg_comp, h, wd, mask, extracted, pred);
    PMS_LAUNCH_CHECK();
  }
  if (labels_out) {
    // rank roots in raster order (scipy.ndimage.label numbering)
    const int gl = std::min(ew_grid(plane), 1024);
    hipLaunchKernelGGL(k_ccl_flatten, dim3(gl, S), dim3(kT), 0, st, lab, (const u64*)bits, h, wd);
    PMS_LAUNCH_CHECK();
    const int chunk = 4096;
    const int nb = (int)((plane + chunk - 1) / chunk);
    uint32_t* counts = nullptr;
    PMS_HIP(hipMallocAsync((void**)&counts, sizeof(uint32_t) * (size_t)S * nb, st));
    int* rank = nullptr;
    PMS_HIP(hipMallocAsync((void**)&rank, sizeof(int) * (size_t)S * plane, st));
    hipLaunchKernelGGL(k_root_count, dim3(nb, S), dim3(kT), 0, st, (const int*)lab, plane, chunk, counts);
    PMS_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_root_scan, dim3(ceil_div(S, 64)), dim3(64), 0, st, counts, nb, S, (uint32_t*)nullptr);
    PMS_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_root_rank, dim3(ceil_div(nb, 64), S), dim3(64), 0, st, lab, plane, chunk,
                       (const uint32_t*)counts, nb, rank);
    PMS_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_label_out, dim3(gl, S), dim3(kT), 0, st, (const int*)lab, (const int*)rank, plane,
                       labels_out);
    PMS_LAUNCH_CHECK();
    PMS_HIP(hipFreeAsync(counts, st));
    PMS_HIP(hipFreeAsync(rank, st));
  }
}
void source_extract(const float* w, int S, int h, int wd, double tol, int neg_comp, uint8_t* mask, float* extracted,
                    int* labels_out, void* work, const int* pred, hipStream_t st) {
  source_extract_t(w, S, h, wd, tol, neg_comp, mask, extracted, labels_out, work, pred, st);
}
void source_extract(const double* w, int S, int h, int wd, double tol, int neg_comp, uint8_t* mask,
                    double* extracted, int* labels_out, void* work, const int* pred, hipStream_t st) {
  source_extract_t(w, S, h, wd, tol, neg_comp, mask, extracted, labels_out, work, pred, st);
}

// ---------------------------------------------------------------- reductions
template <class T>
static void dot_partials_t(const T* a, const T* b, size_t n, double* partial, const int* pred, hipStream_t st) {
  hipLaunchKernelGGL(k_dot<T>, dim3(reduce_grid(n)), dim3(kT), 0, st, a, b, n, partial, pred);
  PMS_LAUNCH_CHECK();
}
void dot_partials(const float* a, const float* b, size_t n, double* partial, const int* pred, hipStream_t st) {
  dot_partials_t(a, b, n, partial, pred, st);
}
void dot_partials(const double* a, const double* b, size_t n, double* partial, const int* pred, hipStream_t st) {
  dot_partials_t(a, b, n, partial, pred, st);
}

void sum_partials(const double* partial, long np, int groups, double* out, const int* pred, hipStream_t st) {
  hipLaunchKernelGGL(k_sum_partials, dim3(groups), dim3(kT), 0, st, partial, np, out, pred);
  PMS_LAUNCH_CHECK();
}

void sum_partials_batch(const SumJob* jobs, int count, hipStream_t st) {
  for (int j0 = 0; j0 < count; j0 += kMaxBatch) {
    const int nb = std::min(kMaxBatch, count - j0);
    SumBatch b{};
    for (int k = 0; k < nb; ++k) {
      b.partial[k] = jobs[j0 + k].partial;
      b.np[k] = jobs[j0 + k].np;
      b.out[k] = jobs[j0 + k].out;
      b.pred[k] = jobs[j0 + k].pred;
    }
    hipLaunchKernelGGL(k_sum_partials_batch, dim3(nb), dim3(kT), 0, st, b);
    PMS_LAUNCH_CHECK();
  }
}

template <class T>
static void plane_sumsq_partials_t(const T* a, int S, size_t plane, double* partial, const int* pred, hipStream_t st) {
  hipLaunchKernelGGL(k_plane_sumsq<T>, dim3(reduce_grid(plane), S), dim3(kT), 0, st, a, plane, partial, pred);
  PMS_LAUNCH_CHECK();
}
void plane_sumsq_partials(const float* a, int S, size_t plane, double* partial, const int* pred, hipStream_t st) {
  plane_sumsq_partials_t(a, S, plane, partial, pred, st);
}
void plane_sumsq_partials(const double* a, int S, size_t plane, double* partial, const int* pred, hipStream_t st) {
  plane_sumsq_partials_t(a, S, plane, partial, pred, st);
}

template <class T>
static void mean_std_t(const T* a, size_t n, double* partial, double* sum_out, double* dev2_out, hipStream_t st) {
  const int g = reduce_grid(n);
  hipLaunchKernelGGL(k_sum<T>, dim3(g), dim3(kT), 0, st, a, n, partial);
  PMS_LAUNCH_CHECK();
  sum_partials(partial, g, 1, sum_out, nullptr, st);
  hipLaunchKernelGGL(k_dev2<T>, dim3(g), dim3(kT), 0, st, a, n, (const double*)sum_out, partial);
  PMS_LAUNCH_CHECK();
  sum_partials(partial, g, 1, dev2_out, nullptr, st);
}
void mean_std(const float* a, size_t n, double* partial, double* sum_out, double* dev2_out, hipStream_t st) {
  mean_std_t(a, n, partial, sum_out, dev2_out, st);
}
void mean_std(const double* a, size_t n, double* partial, double* sum_out, double* dev2_out, hipStream_t st) {
  mean_std_t(a, n, partial, sum_out, dev2_out, st);
}

}  // namespace pms
