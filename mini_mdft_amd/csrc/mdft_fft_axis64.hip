// The compile-time FFT axis kernels in FP64.
#define MDFT_FFT_AXIS_CT
#include "mdft_fft_ct.hpp"

namespace mdft {
template bool launch_axis_ct<double>(cplx<double>*, const cplx<double>*, int, int, bool, int, long, long, hipStream_t);
}  // namespace mdft
