// The compile-time FFT axis kernels in FP32.
#define MDFT_FFT_AXIS_CT
#include "mdft_fft_ct.hpp"

namespace mdft {
template bool launch_axis_ct<float>(cplx<float>*, const cplx<float>*, int, int, bool, int, long, long, hipStream_t);
}  // namespace mdft
