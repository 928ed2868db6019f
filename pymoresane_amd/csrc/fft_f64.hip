// The float64 precision mode's convolutions on power-of-two frames: the kernels of fft_pow2.h in
// double2, frames up to 8192 (one LDS transform holds a column).  The three passes of a 512^2 image on a 1024 frame
// take 6.6 + 11.3 + 5.7 us; on the mixed-radix kernels, as those were before their steps were compiled, the whole
// convolution took 53 us, now 23.  Error against 80-bit arithmetic (relative rms, frames of 64 / 256 / 1024 / 2048):
// 4.0 / 5.6 / 6.2 / 6.8e-16, 4.9 / 6.1 / 7.3 / 7.7e-16 on the mixed-radix kernels; with every power of a twiddle formed
// from one table value 5.2 / 8.2 / 10.3 / 10.9e-16, and a column pass of 9.7 us.
#include "fft_pow2.h"

namespace pms {
namespace {
Pow2Tables<double2> g_tables;
}  // namespace

template <class TIN>
void pow2_psf_spectrum_f64(const TIN* psf, int q, int p, Cx<double>* spec, Cx<double>* work, hipStream_t st) {
  pow2_psf_spectrum<double2>(psf, q, p, reinterpret_cast<double2*>(spec), reinterpret_cast<double2*>(work),
                             g_tables.get(), st);
}
template void pow2_psf_spectrum_f64<float>(const float*, int, int, Cx<double>*, Cx<double>*, hipStream_t);
template void pow2_psf_spectrum_f64<double>(const double*, int, int, Cx<double>*, Cx<double>*, hipStream_t);

void pow2_conv_batch_f64(const GConvJob<double>* jobs, int count, int n, int p, hipStream_t st) {
  pow2_conv_batch<double2>(jobs, count, n, p, g_tables.get(), st);
}

}  // namespace pms
