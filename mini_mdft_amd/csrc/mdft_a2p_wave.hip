// angl2proj for many points on the compile-time angular grids (see
// mdft_proj.hip for the sums).
#include "mdft_proj_ct.hpp"

#include <algorithm>

namespace mdft {

namespace {

// The points of a field from which a lane per point is faster: a block takes 64 of
// them however few there are, and half of the CUs or more need one.  Microseconds,
// mdft_proj.hip's kernel against this one:
//   mmax 5  FP64 5832 points 20.5 / 19.5, 8000 23.3 / 19.4; FP32 8000 19.0 / 15.4
//   mmax 6  FP64 8000 37.7 / 37.7, 10648 48.6 / 39.2; FP32 5832 23.1 / 24.7, 8000 30.3 / 25.2
//   mmax 4  FP64 8000 16.1 / 16.7, 10648 18.6 / 16.8; FP32 8000 14.0 / 13.9, 10648 16.1 / 14.4
//   mmax 3  FP64 8000 9.7 / 9.6 (mrso 1 14.9 / 15.9), 10648 12.2 / 10.3; FP32 8000
//           8.4 / 9.1 (mrso 1 12.6 / 13.0), 10648 9.6 / 8.7
//   mmax 2  FP64 8000 7.6 / 8.3 (mrso 1 9.9 / 10.4), 10648 9.1 / 8.8; FP32 13824
//           7.5 / 7.7 (mrso 1 9.3 / 9.9), 17576 9.3 / 8.7
long min_points(int mmax, bool fp64) {
  return mmax >= 5 ? 7680 : mmax > 2 || fp64 ? 10240 : 16384;
}

// A block takes 64 consecutive r, one per lane, and its waves share out the
// projections.  For each theta the 64 rows of (phi, psi) values go through LDS
// (read in runs of nphi npsi, which is odd, so that a lane reads its own row
// without bank conflicts); a wave then holds in registers the psi sums X_j of
// its mu2 and, because j and nphi - j have conjugate phases,
//   Y_{+-mup} = X_0 + sum_{j <= mmax} (E_j cos +- i O_j sin),
//   E_j = X_j + X_{nphi - j},  O_j = X_j - X_{nphi - j}
// (the psi sums of the real o likewise), and adds W Y to the sums over theta of
// its projections.  A fifth of the products of one thread per (r, theta, mup,
// mu2) with its operands in LDS, which that kernel spent its time reading:
// 64^3 mmax 5 FP64 483 -> 247 us (1.0 GB, 207 us at the copy rate), FP32 291 ->
// 126 (104 us); 45x36x50 mmax 4 FP32 54 -> 30.  At most 13 sums per wave
// (seven waves at mmax 5): 26 sums 315 us in FP64 (256 registers, one wave per SIMD),
// 21 277, 16 284, 10 284, in FP32 123, 147, 146, 133.  Each role is a whole copy
// of the loop: with the roles inside one loop the compiler kept part of the sums
// in memory (659 us).
template <int MMAX, int MRSO, bool CP>
struct A2pPlan {
  static constexpr int kNmu2 = MMAX / MRSO + 1, kMaxSums = 13, kMaxWaves = 8;
  int base[MMAX + 1];  // canonical index of the first projection of m
  int lo[kMaxWaves][kNmu2], hi[kMaxWaves][kNmu2];  // |mup| of a wave at one mu2, empty if lo > hi
  int waves, sums;     // sums: the most projections of one wave
  static constexpr int projections(int b, int a) {  // of (mu2 = b, mup = +-a)
    const int from = a > b * MRSO ? a : b * MRSO;
    return (MMAX - from + 1) * (a == 0 || (CP && b == 0) ? 1 : 2);
  }
  constexpr A2pPlan() : base(), lo(), hi(), waves(0), sums(0) {
    for (int m = 0, n = 0; m <= MMAX; ++m) {
      base[m] = n;
      n += (2 * m + 1) * (m / MRSO + 1);
    }
    int total = 0;
    for (int b = 0; b < kNmu2; ++b)
      for (int a = 0; a <= MMAX; ++a) total += projections(b, a);
    // the fewest waves, from two, whose shares (consecutive (mu2, |mup|), as
    // even as they come) have at most kMaxSums projections
    for (waves = 2;; ++waves) {
      int share[kMaxWaves] = {}, n = 0;
      for (int w = 0; w < waves; ++w)
        for (int b = 0; b < kNmu2; ++b) {
          lo[w][b] = MMAX + 1;
          hi[w][b] = -1;
        }
      for (int b = 0; b < kNmu2; ++b)
        for (int a = 0; a <= MMAX; ++a) {
          const int c = projections(b, a), w = (2 * n + c) * waves / (2 * total);
          if (lo[w][b] > a) lo[w][b] = a;
          hi[w][b] = a;
          share[w] += c;
          n += c;
        }
      sums = 0;
      for (int w = 0; w < waves; ++w)
        if (share[w] > sums) sums = share[w];
      if (sums <= kMaxSums || waves == kMaxWaves) break;
    }
  }
};

// the twiddles of a wave, in scalar registers
template <int MMAX, int MRSO, typename TC>
struct A2pTwiddles {
  static constexpr int kNpsi = 2 * (MMAX / MRSO) + 1, kHalf = kNpsi / 2;
  cplx<TC> phi[MMAX + 1], psi[kHalf + 1];  // e^{2 pi i t/nphi}, e^{2 pi i t/npsi}
};

// adds one theta's terms to the sums of wave W's projections; row: the lane's
// (phi, psi) values, w: the weights of theta
template <int MMAX, int MRSO, bool CP, int W, typename TC, int SUMS>
__device__ __forceinline__ void a2p_wave_theta(const TC* row, const A2pTwiddles<MMAX, MRSO, TC>& tw, const TC* w,
                                               TC (&sr)[SUMS], TC (&si)[SUMS]) {
  using Z = A2pSizes<MMAX, MRSO, 1>;
  constexpr int NPHI = Z::kNphi, NMU2 = Z::kNmu2, NPSI = Z::kNpsi;
  constexpr A2pPlan<MMAX, MRSO, CP> P{};
  int c = 0;
#pragma unroll
  for (int b = 0; b < NMU2; ++b) {
    if (P.lo[W][b] > P.hi[W][b]) continue;
    TC xr[NPHI], xi[NPHI];
#pragma unroll
    for (int j = 0; j < NPHI; ++j) {
      xr[j] = row[j * NPSI];
      xi[j] = 0;
#pragma unroll
      for (int k = 1; 2 * k < NPSI; ++k) {
        const TC u = row[j * NPSI + k], v = row[j * NPSI + NPSI - k];
        if (b == 0) {
          xr[j] += u + v;
        } else {
          const int t = (b * k) % NPSI;
          const cplx<TC> e = tw.psi[2 * t > NPSI ? NPSI - t : t];
          xr[j] = fma(u + v, e.x, xr[j]);
          xi[j] = fma(u - v, 2 * t > NPSI ? -e.y : e.y, xi[j]);
        }
      }
      if (j % 3 == 2) __builtin_amdgcn_sched_barrier(0);  // no more of the row in registers at once
    }
#pragma unroll
    for (int j = 1; j <= MMAX; ++j) {  // E_j in place of X_j, O_j of X_{nphi - j}
      const TC ur = xr[j], ui = xi[j], vr = xr[NPHI - j], vi = xi[NPHI - j];
      xr[j] = ur + vr;
      xi[j] = ui + vi;
      xr[NPHI - j] = ur - vr;
      xi[NPHI - j] = ui - vi;
    }
#pragma unroll
    for (int a = 0; a <= MMAX; ++a) {
      if (a < P.lo[W][b] || a > P.hi[W][b]) continue;
      TC er = xr[0], ei = xi[0], dr = 0, di = 0;
#pragma unroll
      for (int j = 1; j <= MMAX; ++j) {
        const int t = (a * j) % NPHI;  // the twiddles of t and nphi - t are conjugate
        const cplx<TC> e = tw.phi[t > MMAX ? NPHI - t : t];
        const TC sn = t > MMAX ? -e.y : e.y;
        er = a == 0 ? er + xr[j] : fma(xr[j], e.x, er);
        if (a > 0) dr = fma(xr[NPHI - j], sn, dr);
        if (b > 0) {
          ei = a == 0 ? ei + xi[j] : fma(xi[j], e.x, ei);
          if (a > 0) di = fma(xi[NPHI - j], sn, di);
        }
      }
#pragma unroll
      for (int g = 0; g < 2; ++g) {  // mup = a, -a
        if (g == 1 && (a == 0 || (CP && b == 0))) continue;
        const int mup = g ? -a : a;
        const TC yr = g ? er + di : er - di, yi = g ? ei - dr : ei + dr;
#pragma unroll
        for (int m = 0; m <= MMAX; ++m) {
          if (m < a || m < b * MRSO) continue;
          const TC wv = w[P.base[m] + (mup + m) * (m / MRSO + 1) + b];
          sr[c] = fma(wv, yr, sr[c]);
          si[c] = fma(wv, yi, si[c]);
          ++c;
        }
      }
    }
  }
}

// writes wave W's sums, in the order of a2p_wave_theta, to point r
template <int MMAX, int MRSO, bool CP, int W, typename TP, typename TC, int SUMS>
__device__ __forceinline__ void a2p_wave_store(cplx<TP>* __restrict__ p, long N, long r, const TC (&sr)[SUMS],
                                               const TC (&si)[SUMS]) {
  constexpr A2pPlan<MMAX, MRSO, CP> P{};
  constexpr CompactMap<MMAX, MRSO> kCm{};
  int c = 0;
#pragma unroll
  for (int b = 0; b < A2pPlan<MMAX, MRSO, CP>::kNmu2; ++b)
#pragma unroll
    for (int a = 0; a <= MMAX; ++a) {
      if (a < P.lo[W][b] || a > P.hi[W][b]) continue;
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        if (g == 1 && (a == 0 || (CP && b == 0))) continue;
#pragma unroll
        for (int m = 0; m <= MMAX; ++m) {
          if (m < a || m < b * MRSO) continue;
          const int ip = P.base[m] + ((g ? -a : a) + m) * (m / MRSO + 1) + b;
          p[static_cast<long>(CP ? kCm.v[ip] : ip) * N + r] = mkc<TP>(static_cast<TP>(sr[c]), static_cast<TP>(si[c]));
          ++c;
        }
      }
    }
}

// wave W of a block (each wave of the block passes the same barriers)
template <int MMAX, int MRSO, bool CP, int W, typename TI, typename TP, typename TC>
__device__ __forceinline__ void a2p_wave(const TI* __restrict__ o, cplx<TP>* __restrict__ p, long N,
                                         const TabPtrs<TC>& tb, int fuse, double rho0, TC* stage, TC* wts) {
  using Z = A2pSizes<MMAX, MRSO, 1>;
  constexpr A2pPlan<MMAX, MRSO, CP> P{};
  constexpr int NJK = Z::kNphi * Z::kNpsi, NO = Z::kNo, NTH = Z::kNth, NP = Z::kNp();
  constexpr int kT = 64 * P.waves, kPer = (64 * NJK + kT - 1) / kT;
  const int tid = threadIdx.x, lane = tid & 63;
  const long r0 = static_cast<long>(blockIdx.x) * 64;
  const int last = static_cast<int>(min(63L, N - 1 - r0));  // rows past the end repeat the last one
  const TI* src = o + r0 * NO;
  A2pTwiddles<MMAX, MRSO, TC> tw;
#pragma unroll
  for (int t = 0; t <= MMAX; ++t) tw.phi[t] = tb.ephi[t];
#pragma unroll
  for (int t = 0; t <= tw.kHalf; ++t) tw.psi[t] = tb.epsi[(MMAX >= MRSO ? Z::kNpsi : 0) + t];
  TC sr[P.sums], si[P.sums];
#pragma unroll
  for (int i = 0; i < P.sums; ++i) sr[i] = si[i] = 0;
  unsigned off[kPer];  // bytes
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int e = min(tid + u * kT, 64 * NJK - 1), row = e / NJK;
    off[u] = (min(row, last) * NO + (e - row * NJK)) * sizeof(TI);
  }
  TI v[kPer];
  const auto request = [&](int th) {
    const char* from = reinterpret_cast<const char*>(src + th * NJK);
#pragma unroll
    for (int u = 0; u < kPer; ++u) v[u] = *reinterpret_cast<const TI*>(from + off[u]);
  };
  request(0);
  for (int i = tid; i < NTH * NP; i += kT) wts[i] = tb.wts[i];
#pragma unroll 1
  for (int th = 0; th < NTH; ++th) {
    if (th > 0) __syncthreads();  // the waves have read the previous theta
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int e = tid + u * kT;
      const double x = static_cast<double>(v[u]);
      if (e < 64 * NJK) stage[e] = static_cast<TC>(fuse ? rho0 * (x * x - 1.0) : x);
    }
    request(min(th + 1, NTH - 1));
    __syncthreads();
    a2p_wave_theta<MMAX, MRSO, CP, W>(stage + lane * NJK, tw, wts + th * NP, sr, si);
  }
  if (lane <= last) a2p_wave_store<MMAX, MRSO, CP, W, TP>(p, N, r0 + lane, sr, si);
}

template <int MMAX, int MRSO, typename TI, typename TP, typename TC, bool CP>
__global__ __launch_bounds__((64 * A2pPlan<MMAX, MRSO, CP>().waves)) void angl2proj_wave_kernel(
    const TI* __restrict__ o, cplx<TP>* __restrict__ p, long N, TabPtrs<TC> tb, int fuse, double rho0) {
  using Z = A2pSizes<MMAX, MRSO, 1>;
  constexpr A2pPlan<MMAX, MRSO, CP> P{};
  __shared__ TC stage[64 * Z::kNphi * Z::kNpsi];
  __shared__ TC wts[Z::kNth * Z::kNp()];
  dispatch_wave<P.waves>(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6), [&](auto ww) {
    a2p_wave<MMAX, MRSO, CP, decltype(ww)::value, TI, TP, TC>(o, p, N, tb, fuse, rho0, stage, wts);
  });
}

}  // namespace

template <typename TI, typename TP, typename TC>
bool launch_a2p_wave(const ProjTables& t, long N, long field, const TI* o, cplx<TP>* p, const TabPtrs<TC>& tb,
                     const double* drho_rho0, hipStream_t s, bool compact) {
  if (field < min_points(t.mmax, std::is_same<TC, double>::value)) return false;
  bool done = false;
  dispatch_angular(t.mmax, t.mrso, [&](auto mm, auto mr) {
    constexpr int MMAX = decltype(mm)::value, MRSO = decltype(mr)::value;
    if constexpr (MMAX >= 2) {
      auto go = [&](auto kernel, int waves) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>((N + 63) / 64)), dim3(64 * waves), 0, s, o, p, N, tb,
                           drho_rho0 ? 1 : 0, drho_rho0 ? *drho_rho0 : 0.0);
        MDFT_HIP_CHECK(hipGetLastError());
        done = true;
      };
      if (compact)
        go(angl2proj_wave_kernel<MMAX, MRSO, TI, TP, TC, true>, A2pPlan<MMAX, MRSO, true>().waves);
      else
        go(angl2proj_wave_kernel<MMAX, MRSO, TI, TP, TC, false>, A2pPlan<MMAX, MRSO, false>().waves);
    }
  });
  return done;
}

template bool launch_a2p_wave<double, double, double>(const ProjTables&, long, long, const double*, cplx<double>*,
                                                      const TabPtrs<double>&, const double*, hipStream_t, bool);
template bool launch_a2p_wave<float, float, float>(const ProjTables&, long, long, const float*, cplx<float>*,
                                                   const TabPtrs<float>&, const double*, hipStream_t, bool);

}  // namespace mdft
