// Entry points of the FFT convolution in float32: power-of-two frames on the kernels of fft_pow2.h,
// other even frames on the mixed-radix ones (fft_any.hip).  Reference:
// pymoresane/iuwt_convolution.py:18-73.
#include <vector>

#include "fft_pow2.h"

namespace pms {
namespace {
Pow2Tables<float2> g_tables;
}  // namespace

void fft_init_device(int device) { (void)g_tables.get(device); }

int fft_perm(int k, int p) { return is_pow2(p) ? perm_pos(k, ilog2(p)) : gfft_perm(k, p); }

size_t fft_spectrum_elems(int p) { return (size_t)(p / 2 + 1) * p; }

size_t fft_conv_work_elems(int n, int p) { return 2 * (size_t)(p / 2 + 1) * n; }

static void check_fft_len(int p) {
  PMS_REQUIRE(is_pow2(p) && p >= 4 && p <= kFftMaxLen,
              "FFT frame side must be a power of two in [4, " + std::to_string(kFftMaxLen) +
                  "], got " + std::to_string(p));
}

void fft_psf_spectrum(const float* psf, int q, int p, float2* spec, float2* work, hipStream_t st) {
  if (!is_pow2(p)) {
    // any other even side: the mixed-radix transforms (same layout, digit-reversed columns)
    gfft_psf_spectrum<float, float>(psf, q, p, reinterpret_cast<Cx<float>*>(spec), reinterpret_cast<Cx<float>*>(work),
                                    st);
    return;
  }
  check_fft_len(p);
  PMS_REQUIRE(q >= 1 && q <= p, "PSF larger than the FFT frame");
  pow2_psf_spectrum<float2>(psf, q, p, spec, work, g_tables.get(), st);
}

void fft_conv(const float* in, int n, int p, const float2* spec, float* out, float2* work, const int* pred,
              hipStream_t st) {
  const FftConvJob j{in, spec, out, work, pred};
  fft_conv_batch(&j, 1, n, p, st);
}

void fft_conv_batch(const FftConvJob* jobs, int count, int n, int p, hipStream_t st) {
  if (!is_pow2(p)) {
    std::vector<GConvJob<float>> g(count);
    for (int k = 0; k < count; ++k)
      g[k] = GConvJob<float>{jobs[k].in, reinterpret_cast<const Cx<float>*>(jobs[k].spec), jobs[k].out,
                             reinterpret_cast<Cx<float>*>(jobs[k].work), jobs[k].pred};
    gfft_conv_batch<float>(g.data(), count, n, p, st);
    return;
  }
  check_fft_len(p);
  pow2_conv_batch<float2>(jobs, count, n, p, g_tables.get(), st);
}

// numpy rfft2 spectrum (rows = axis-0 frequency m in [0,P), cols = k in [0,P/2]) of an
// unrolled PSF frame -> library layout: column k, position perm(m), times (-1)^(m+k)
// (the P/2 roll in both axes).
void fft_spectrum_from_numpy_host(const float* re_im, int p, float2* spec_host) {
  if (is_pow2(p))
    check_fft_len(p);
  else
    PMS_REQUIRE(gfft_frame_ok(p, sizeof(float)), "FFT frame side " + std::to_string(p) + " is not supported");
  const int nk = p / 2 + 1;
  for (int m = 0; m < p; ++m) {
    const int pos = fft_perm(m, p);
    for (int k = 0; k < nk; ++k) {
      const float sgn = ((m + k) & 1) ? -1.f : 1.f;
      const float* v = re_im + 2 * ((size_t)m * nk + k);
      spec_host[(size_t)k * p + pos] = make_float2(sgn * v[0], sgn * v[1]);
    }
  }
}

}  // namespace pms
