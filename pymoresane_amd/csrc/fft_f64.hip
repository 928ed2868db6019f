// The float64 precision mode's convolutions on power-of-two frames: the kernels of fft_pow2.h in
// double2, frames up to 8192 (one LDS transform holds a column).  On a 1024 frame the three passes take
// 5.6 + 9.0 + 5.4 us, where the mixed-radix kernels, whose plan, digit reversal and twiddle reads are worked out
// at run time, take 17.1 + 18.0 + 11.3 us.
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
