// What the kernels for compile-time angular grids share (mdft_proj.hip,
// mdft_a2p_wave.hip, mdft_p2a_wave.hip).
#pragma once

#include <type_traits>

#include "mdft_proj.hpp"

namespace mdft {

template <typename TC>
struct TabPtrs {
  const cplx<TC>* ephi;
  const cplx<TC>* epsi;
  const TC* wts;
  const int* ipinfo;
  const int* yidx;
};

template <int MMAX, int MRSO, int RT>
struct A2pSizes {
  static constexpr int kNth = MMAX + 1, kNphi = 2 * MMAX + 1, kNmu2 = MMAX / MRSO + 1;
  static constexpr int kNpsi = 2 * (MMAX / MRSO) + 1, kNo = kNth * kNphi * kNpsi;
  static constexpr int kNp() {
    int n = 0;
    for (int m = 0; m <= MMAX; ++m) n += (2 * m + 1) * (m / MRSO + 1);
    return n;
  }
  static constexpr int kCells = RT * kNth * kNphi * kNmu2;
  static constexpr int kRegA = (2 * kCells > RT * kNo) ? 2 * kCells : RT * kNo;
};

// the angular grids with a compile-time proj2angl kernel: mrso = 2 with mmax
// 1..6 and mrso = 1 with mmax 1..3 (larger mrso = 1 grids hold too many S
// registers per lane and take the generic kernel)
template <int MMAX = 1, int MRSO = 1, typename F>
bool dispatch_angular(int mmax, int mrso, F&& f) {
  if constexpr (MMAX > 6) {
    return false;
  } else if constexpr (MRSO > 2 || (MRSO == 1 && MMAX > 3)) {
    return dispatch_angular<MMAX + (MRSO > 2 ? 1 : 0), MRSO + (MRSO > 2 ? -2 : 1)>(mmax, mrso, f);
  } else {
    if (mmax == MMAX && mrso == MRSO) {
      f(std::integral_constant<int, MMAX>{}, std::integral_constant<int, MRSO>{});
      return true;
    }
    return dispatch_angular<MMAX, MRSO + 1>(mmax, mrso, f);
  }
}

// f(integral_constant<int, w>) for the wave-uniform w < N
template <int N, int W = 0, typename F>
__device__ __forceinline__ void dispatch_wave(int w, F&& f) {
  if constexpr (W + 1 == N) {
    f(std::integral_constant<int, W>{});
  } else {
    if (w == W)
      f(std::integral_constant<int, W>{});
    else
      dispatch_wave<N, W + 1>(w, f);
  }
}

// angl2proj with one point per lane (mdft_a2p_wave.hip); false if the grid or
// the number of points of a field is not one it serves
template <typename TI, typename TP, typename TC>
bool launch_a2p_wave(const ProjTables& t, long N, long field, const TI* o, cplx<TP>* p, const TabPtrs<TC>& tb,
                     const double* drho_rho0, hipStream_t s, bool compact);

// proj2angl with a wave per mu2 (mdft_p2a_wave.hip); false if the grid is not one
// it serves
template <typename TP, typename TO, typename TC>
bool launch_p2a_wave(const ProjTables& t, long N, const cplx<TP>* p, TO* o, const TO* xi, TO* df,
                     const TabPtrs<TC>& tb, double rho0, double* partials, hipStream_t s, double* colpart, bool compact);

}  // namespace mdft
