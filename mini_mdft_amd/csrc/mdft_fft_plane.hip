// The compile-time FFT plane kernels: z and y of an n x n plane in one pass.
#include "mdft_fft_ct.hpp"

namespace mdft {

namespace {

// plane_ct at compile time
template <typename T, int N>
constexpr bool plane_fits() {
  return plane_ct_bytes(N, sizeof(cplx<T>)) <= kLdsMax;
}
// The lengths whose planes are compiled with 256 and with 512 threads (the
// tuner's choice).  The others have one count: up to 32 a stage has at most 256
// butterflies of radix 4 and a block of 512 would idle; above, 512 threads keep
// eight waves on a CU where only one or two planes fit in its LDS.
constexpr bool both_threads(int n) {
  return n == 16 || n == 32 || n == 48 || n == 64 || n == 80 || n == 96;
}

}  // namespace

template <typename T>
bool launch_plane_ct(cplx<T>* data, const cplx<T>* tw, int n, long planes, int threads, int sign, hipStream_t s) {
  bool done = false;
  for_length(n, CtLengths{}, [&](auto nn) {
    constexpr int N = decltype(nn)::value;
    if constexpr (plane_fits<T, N>()) {
      constexpr size_t lds = plane_ct_bytes(N, sizeof(cplx<T>));
      auto go = [&](auto kernel, int th) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(planes)), dim3(th), lds, s, data, tw, sign);
        MDFT_HIP_CHECK(hipGetLastError());
        done = true;
      };
      if constexpr (both_threads(N)) {
        if (threads == 256)
          go(fft_plane_ct_kernel<T, N, 256>, 256);
        else
          go(fft_plane_ct_kernel<T, N, 512>, 512);
      } else {
        constexpr int th = N <= 32 ? 256 : 512;
        go(fft_plane_ct_kernel<T, N, th>, th);
      }
    }
  });
  return done;
}

template bool launch_plane_ct<float>(cplx<float>*, const cplx<float>*, int, long, int, int, hipStream_t);
template bool launch_plane_ct<double>(cplx<double>*, const cplx<double>*, int, long, int, int, hipStream_t);

}  // namespace mdft
