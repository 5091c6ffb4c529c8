// The compile-time FFT plane kernels: z and y of an n x n plane in one pass.
#include "mdft_fft_ct.hpp"

namespace mdft {

namespace {

// plane_ct at compile time
template <typename T, int N>
constexpr bool plane_fits() {
  return plane_ct_bytes(N, sizeof(cplx<T>)) <= kLdsMax;
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
        constexpr int th = plane_ct_threads(N, 0);
        go(fft_plane_ct_kernel<T, N, th>, th);
      }
    }
  });
  return done;
}

template bool launch_plane_ct<float>(cplx<float>*, const cplx<float>*, int, long, int, int, hipStream_t);
template bool launch_plane_ct<double>(cplx<double>*, const cplx<double>*, int, long, int, int, hipStream_t);

}  // namespace mdft
