// Compile-time kernels of the 3D FFT (see mdft_fft.hip): the butterflies, and
// the axis and plane kernels for fixed lengths.  Included by the translation
// units that instantiate them (mdft_fft_axis32.hip, mdft_fft_axis64.hip,
// mdft_fft_plane.hip) and by mdft_fft.hip for its run-time kernels.
#pragma once

#include <type_traits>
#include <utility>

#include "mdft_fft.hpp"

namespace mdft {

constexpr int kFftThreads = 256;
constexpr int kMaxRadix = 13;
constexpr size_t kLdsMax = 160 * 1024;

template <typename T>
__device__ __forceinline__ cplx<T> twiddle(const cplx<T>* tw, int t, int sign) {
  cplx<T> w = tw[t];
  if (sign > 0) w.y = -w.y;
  return w;
}

// x * w with one fused and one rounded product, written out so that every
// kernel (run-time or compile-time stages, any tiling) rounds the same way
// whatever the compiler would contract
template <typename T>
__device__ __forceinline__ cplx<T> tw_mul(cplx<T> x, cplx<T> w) {
  return mkc<T>(fma(x.x, w.x, -(x.y * w.y)), fma(x.x, w.y, x.y * w.x));
}

// in-place DFT of R values; sign -1 forward, +1 backward
template <typename T>
__device__ __forceinline__ void dft_small(cplx<T>* v, int R, int sign, const cplx<T>* tw, int n) {
  if (R == 2) {
    cplx<T> a = v[0], b = v[1];
    v[0] = cadd<T>(a, b);
    v[1] = csub<T>(a, b);
  } else if (R == 4) {
    cplx<T> s02 = cadd<T>(v[0], v[2]), d02 = csub<T>(v[0], v[2]);
    cplx<T> s13 = cadd<T>(v[1], v[3]), d13 = csub<T>(v[1], v[3]);
    // W = e^{sign 2 pi i/4} = sign * i
    cplx<T> wd = mkc<T>(-static_cast<T>(sign) * d13.y, static_cast<T>(sign) * d13.x);
    v[0] = cadd<T>(s02, s13);
    v[2] = csub<T>(s02, s13);
    v[1] = cadd<T>(d02, wd);
    v[3] = csub<T>(d02, wd);
  } else if (R == 3) {
#pragma clang fp contract(off)
    const T h = static_cast<T>(0.86602540378443864676);  // sqrt(3)/2
    cplx<T> a = v[0], t = cadd<T>(v[1], v[2]), u = csub<T>(v[1], v[2]);
    cplx<T> m = mkc<T>(a.x - static_cast<T>(0.5) * t.x, a.y - static_cast<T>(0.5) * t.y);
    // sign * i * h * u
    cplx<T> r = mkc<T>(-static_cast<T>(sign) * h * u.y, static_cast<T>(sign) * h * u.x);
    v[0] = cadd<T>(a, t);
    v[1] = cadd<T>(m, r);
    v[2] = csub<T>(m, r);
  } else {
    cplx<T> out[kMaxRadix];
    const int step = n / R;
    for (int s = 0; s < R; ++s) {
      cplx<T> acc = v[0];
      for (int r = 1; r < R; ++r) acc = cfma<T>(acc, v[r], twiddle<T>(tw, ((r * s) % R) * step, sign));
      out[s] = acc;
    }
    for (int s = 0; s < R; ++s) v[s] = out[s];
  }
}

// DFT of R values held in registers (R fixed at compile time)
template <typename T, int R>
__device__ __forceinline__ void dft_fixed(cplx<T> (&v)[R], int sign, const cplx<T>* tw, int n) {
  if constexpr (R == 2 || R == 3 || R == 4) {
    dft_small<T>(v, R, sign, tw, n);
  } else {
    cplx<T> out[R];
    const int step = n / R;
#pragma unroll
    for (int s = 0; s < R; ++s) {
      cplx<T> acc = v[0];
#pragma unroll
      for (int r = 1; r < R; ++r) acc = cfma<T>(acc, v[r], twiddle<T>(tw, ((r * s) % R) * step, sign));
      out[s] = acc;
    }
#pragma unroll
    for (int s = 0; s < R; ++s) v[s] = out[s];
  }
}

// Lengths with compile-time kernels: 8 .. 128 with prime factors up to 13, in
// the radix schedule of FftPlan1D (4s first, then 2, 3, 5, 7, 11, 13).  Each
// stage has its length, strides, line and thread counts known at compile time,
// so the index arithmetic reduces to shifts, masks and constant divisions and
// the butterfly loop unrolls; the arithmetic of every butterfly (LDS twiddles,
// run-time sign, explicitly rounded products, operation order) is that of the
// run-time stages, so results are bitwise the same.  The run-time kernels spend
// most of their time on divisions by run-time lengths and on odd primes.  One
// 3D transform of the 73 channels of mmax 5 (45 of mmax 4 at 45x36x50 and 56^3),
// run-time stages against these, microseconds:
//   FP32  96^3 829 -> 576, 80^3 416 -> 330, 4 x 48^3 261 -> 185, 40^3 73 -> 43,
//         56^3 246 -> 65, 45x36x50 61 -> 52
//   FP64  80^3 948 -> 686, 48^3 126 -> 104
// (64^3 and 32^3 had compiled kernels already and are the same).  The bytes are
// two round trips of the channels: 96^3 2.07 GB, 430 us at the copy rate.
template <int... N>
struct Lengths {};
using CtLengths =
    Lengths<8, 9, 10, 11, 12, 13, 14, 15, 16, 18, 20, 21, 22, 24, 25, 26, 27, 28, 30, 32, 33, 35, 36, 39, 40, 42, 44, 45,
            48, 49, 50, 52, 54, 55, 56, 60, 63, 64, 65, 66, 70, 72, 75, 77, 78, 80, 81, 84, 88, 90, 91, 96, 98, 99, 100,
            104, 105, 108, 110, 112, 117, 120, 121, 125, 126, 128>;

// f(integral_constant<int, n>) if n is one of the lengths
template <typename F, int... N>
bool for_length(int n, Lengths<N...>, F&& f) {
  return ((n == N ? (f(std::integral_constant<int, N>{}), true) : false) || ...);
}
inline bool ct_length(int n) {
  return for_length(n, CtLengths{}, [](auto) {});
}

template <int N>
constexpr int ct_nstages() {
  constexpr int ps[7] = {4, 2, 3, 5, 7, 11, 13};
  int r = N, c = 0;
  for (int p : ps)
    while (r % p == 0) {
      r /= p;
      ++c;
    }
  return c;
}
template <int N>
constexpr int ct_radix(int s) {
  constexpr int ps[7] = {4, 2, 3, 5, 7, 11, 13};
  int r = N, c = 0;
  for (int p : ps)
    while (r % p == 0) {
      if (c == s) return p;
      r /= p;
      ++c;
    }
  return 0;
}
// Lines per tile of the contiguous axis: 8 KB of values, and at most 64 (one pass
// over 73 x 64^3 values, us, tiles of 4 / 8 / 16 KB: FP32 64-long lines 43 / 38 /
// 39, 45 53 / 48 / 55, 96 56 / 49 / 57; FP64 64 86 (8) / 88 (16), 45 100 / 130, 96 102 / 132).
template <typename T>
constexpr int contiguous_lines(int n) {
  const int w = 8192 / static_cast<int>(sizeof(cplx<T>)) / n;
  return w < 64 ? w : 64;
}
// Tiles of a strided axis: 16 neighbouring columns and, for short lines, 32 or 64,
// for long ones 8, which some fields need to fill the chip (9 x 128 x 32 x 64
// FP32, y and x: 16 columns 38 us, 8 37; 1168 x 128 x 16 27.6 against 22.3), and 4
// (strides below 8).  They need not divide the stride: a last tile with missing
// columns costs one part in the number of tiles, while a width that had to
// divide it left 48^2 and 96^2 to the run-time kernel (4 x 48^3: 175 us for the
// x axis alone, now 97).
constexpr bool strided_lines(int n, int w) {
  return w == 16 || (w == 32 && n <= 64) || (w == 64 && n <= 32) || ((w == 4 || w == 8) && n >= 64);
}

template <typename T, int R, int N, int NS, int LS, int ES, int NLINES, int NTH, bool W_FAST>
__device__ __forceinline__ void ct_stage_2d(const cplx<T>* src, cplx<T>* dst, const cplx<T>* tw, int sign, int tid) {
  constexpr int NB = N / R, TSTEP = N / (NS * R), TOTAL = NLINES * NB;
  constexpr int ITERS = (TOTAL + NTH - 1) / NTH;
#pragma unroll
  for (int i = 0; i < ITERS; ++i) {
    const int beta = tid + i * NTH;
    if (TOTAL % NTH == 0 || beta < TOTAL) {
      int w, j;
      if constexpr (W_FAST) {
        j = beta / NLINES;
        w = beta - j * NLINES;
      } else {
        w = beta / NB;
        j = beta - w * NB;
      }
      const int k = j % NS;
      const cplx<T>* in = src + w * LS + j * ES;
      cplx<T> v[R];
      v[0] = in[0];
#pragma unroll
      for (int r = 1; r < R; ++r) v[r] = tw_mul<T>(in[r * NB * ES], twiddle<T>(tw, r * k * TSTEP, sign));
      dft_fixed<T, R>(v, sign, tw, N);
      cplx<T>* out = dst + w * LS + ((j / NS) * NS * R + k) * ES;
#pragma unroll
      for (int r = 0; r < R; ++r) out[r * NS * ES] = v[r];
    }
  }
}

// stages S.. of one axis over an LDS tile, ping-pong between a and b; the
// result ends in a when the remaining stage count is even, else in b
template <typename T, int N, int LS, int ES, int NLINES, int NTH, bool W_FAST, int S = 0, int NS = 1>
__device__ __forceinline__ void ct_stockham_2d(cplx<T>* a, cplx<T>* b, const cplx<T>* tw, int sign, int tid) {
  if constexpr (S < ct_nstages<N>()) {
    constexpr int R = ct_radix<N>(S);
    ct_stage_2d<T, R, N, NS, LS, ES, NLINES, NTH, W_FAST>(a, b, tw, sign, tid);
    __syncthreads();
    ct_stockham_2d<T, N, LS, ES, NLINES, NTH, W_FAST, S + 1, NS * R>(b, a, tw, sign, tid);
  }
}

// One stage of the lines of an LDS tile in place: every butterfly of the block in
// registers between two barriers.
template <typename T, int R, int N, int NS, int LS, int ES, int NLINES, int NTH, bool W_FAST>
__device__ __forceinline__ void ct_stage_in_place(cplx<T>* buf, const cplx<T>* tw, int sign, int tid) {
  constexpr int NB = N / R, TSTEP = N / (NS * R), TOTAL = NLINES * NB;
  constexpr int ITERS = (TOTAL + NTH - 1) / NTH;
  cplx<T> v[ITERS][R];
#pragma unroll
  for (int i = 0; i < ITERS; ++i) {
    const int beta = tid + i * NTH;
    if (TOTAL % NTH == 0 || beta < TOTAL) {
      const int w = W_FAST ? beta % NLINES : beta / NB, j = W_FAST ? beta / NLINES : beta % NB;
      const int k = j % NS;
      const cplx<T>* in = buf + w * LS + j * ES;
      v[i][0] = in[0];
#pragma unroll
      for (int r = 1; r < R; ++r) v[i][r] = tw_mul<T>(in[r * NB * ES], twiddle<T>(tw, r * k * TSTEP, sign));
      dft_fixed<T, R>(v[i], sign, tw, N);
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ITERS; ++i) {
    const int beta = tid + i * NTH;
    if (TOTAL % NTH == 0 || beta < TOTAL) {
      const int w = W_FAST ? beta % NLINES : beta / NB, j = W_FAST ? beta / NLINES : beta % NB;
      cplx<T>* out = buf + w * LS + ((j / NS) * NS * R + j % NS) * ES;
#pragma unroll
      for (int r = 0; r < R; ++r) out[r * NS * ES] = v[i][r];
    }
  }
  __syncthreads();
}

template <typename T, int N, int LS, int ES, int NLINES, int NTH, bool W_FAST, int S = 0, int NS = 1>
__device__ __forceinline__ void ct_stockham_in_place(cplx<T>* buf, const cplx<T>* tw, int sign, int tid) {
  if constexpr (S < ct_nstages<N>()) {
    constexpr int R = ct_radix<N>(S);
    ct_stage_in_place<T, R, N, NS, LS, ES, NLINES, NTH, W_FAST>(buf, tw, sign, tid);
    ct_stockham_in_place<T, N, LS, ES, NLINES, NTH, W_FAST, S + 1, NS * R>(buf, tw, sign, tid);
  }
}

// The plane kernel's stages go back and forth between two padded planes while
// three blocks of those fit on a CU (160 KB), else they work in place on one: a
// block waits for its plane, transforms it, and stores it, and only another
// block on the CU overlaps that.  One 3D transform of the stored channels, two
// planes against one, microseconds: FP32 96^3 (one block a CU against two) 581
// -> 454, 80^3 332 -> 261, 72^3 266 -> 198, 64^3 115 -> 108, FP64 64^3 263 -> 205,
// 80^3 (two axis passes, as two planes do not fit) 662 -> 581.  With three blocks
// and more the extra barrier of a stage is paid for at some lengths only: FP32
// 4 x 48^3 185 -> 175, but 56^3 65 -> 68, 40^3 43 -> 45.
constexpr bool plane_in_place(int n, size_t elem) {
  return (2 * static_cast<size_t>(n) * (n + 1) + n) * elem > kLdsMax / 3;
}
// LDS of the kernel: one or two padded planes and the twiddles
constexpr size_t plane_ct_bytes(int n, size_t elem) {
  return ((plane_in_place(n, elem) ? 1 : 2) * static_cast<size_t>(n) * (n + 1) + n) * elem;
}

// fft_plane_kernel for an N x N plane with NTH threads
template <typename T, int N, int NTH>
__global__ __launch_bounds__(NTH) void fft_plane_ct_kernel(cplx<T>* __restrict__ data, const cplx<T>* __restrict__ tw_g,
                                                           int sign) {
  extern __shared__ unsigned char lds_raw[];
  constexpr int LD = N + 1, NN = N * N, ITERS = (NN + NTH - 1) / NTH;
  constexpr bool kInPlace = plane_in_place(N, sizeof(cplx<T>));
  cplx<T>* buf = reinterpret_cast<cplx<T>*>(lds_raw);
  cplx<T>* tw = buf + (kInPlace ? 1 : 2) * N * LD;
  const int tid = threadIdx.x;
  if (tid < N) tw[tid] = tw_g[tid];
  cplx<T>* plane = data + static_cast<long>(blockIdx.x) * NN;
#pragma unroll
  for (int i = 0; i < ITERS; ++i) {
    const int t = tid + i * NTH;
    if (NN % NTH == 0 || t < NN) buf[(t / N) * LD + t % N] = plane[t];
  }
  __syncthreads();
  // z along the rows, then y along the columns
  if constexpr (kInPlace) {
    ct_stockham_in_place<T, N, LD, 1, N, NTH, false>(buf, tw, sign, tid);
    ct_stockham_in_place<T, N, 1, LD, N, NTH, true>(buf, tw, sign, tid);
  } else {  // two axes of the same stage count end where they began
    cplx<T>* second = buf + N * LD;
    constexpr bool odd = ct_nstages<N>() % 2 == 1;
    ct_stockham_2d<T, N, LD, 1, N, NTH, false>(buf, second, tw, sign, tid);
    ct_stockham_2d<T, N, 1, LD, N, NTH, true>(odd ? second : buf, odd ? buf : second, tw, sign, tid);
  }
#pragma unroll
  for (int i = 0; i < ITERS; ++i) {
    const int t = tid + i * NTH;
    if (NN % NTH == 0 || t < NN) plane[t] = buf[(t / N) * LD + t % N];
  }
}

// fft_axis_kernel for length N and tiles of W lines, nchunk of them in a strided
// row of S columns.  The last tile may be ragged: its missing lines are computed
// on and not stored.  Whole tiles have a branch of their own, whose loads are
// requested together: a test of each value against the end of the data took
// the 64-long FP64 lines of 73 x 64^3 values from 86 to 113 us, FP32 from 38 to 42.
template <typename T, bool STRIDED, int N, int W>
__global__ __launch_bounds__(kFftThreads) void fft_axis_ct_kernel(cplx<T>* __restrict__ data,
                                                                  const cplx<T>* __restrict__ tw_g, int sign,
                                                                  long nlines, long S, unsigned nchunk) {
  extern __shared__ unsigned char lds_raw[];
  constexpr int LD = N + 1, NTH = kFftThreads, WN = W * N, ITERS = (WN + NTH - 1) / NTH;
  cplx<T>* bufA = reinterpret_cast<cplx<T>*>(lds_raw);
  cplx<T>* bufB = bufA + W * LD;
  cplx<T>* tw = bufB + W * LD;
  const int tid = threadIdx.x;
  if (tid < N) tw[tid] = tw_g[tid];
  long base;
  int valid;  // lines of this tile
  if constexpr (!STRIDED) {
    const long l0 = static_cast<long>(blockIdx.x) * W;
    base = l0 * N;
    valid = static_cast<int>(min(static_cast<long>(W), nlines - l0));
  } else {
    const unsigned o = blockIdx.x / nchunk;
    const long i0 = static_cast<long>(blockIdx.x - o * nchunk) * W;
    base = static_cast<long>(o) * N * S + i0;
    valid = static_cast<int>(min(static_cast<long>(W), S - i0));
  }
  // value i of this thread: its place in the tile's data, and in LDS
  const auto from = [&](int i) {
    const int t = tid + i * NTH;
    return base + (STRIDED ? static_cast<long>(t / W) * S + t % W : t);
  };
  const auto to = [&](int i) {
    const int t = tid + i * NTH;
    return STRIDED ? (t % W) * LD + t / W : (t / N) * LD + t % N;
  };
  const auto in_tile = [&](int i) { return WN % NTH == 0 || tid + i * NTH < WN; };
  const auto exists = [&](int i) {
    const int t = tid + i * NTH;
    return in_tile(i) && (STRIDED ? t % W : t / N) < valid;
  };
  if (valid == W) {
#pragma unroll
    for (int i = 0; i < ITERS; ++i)
      if (in_tile(i)) bufA[to(i)] = data[from(i)];
  } else {
#pragma unroll 1
    for (int i = 0; i < ITERS; ++i)
      if (exists(i)) bufA[to(i)] = data[from(i)];
  }
  __syncthreads();
  ct_stockham_2d<T, N, LD, 1, W, NTH, false>(bufA, bufB, tw, sign, tid);
  const cplx<T>* res = ct_nstages<N>() % 2 == 0 ? bufA : bufB;
  if (valid == W) {
#pragma unroll
    for (int i = 0; i < ITERS; ++i)
      if (in_tile(i)) data[from(i)] = res[to(i)];
  } else {
#pragma unroll 1
    for (int i = 0; i < ITERS; ++i)
      if (exists(i)) data[from(i)] = res[to(i)];
  }
}

template <typename T>
constexpr size_t axis_lds(int n, int W) {
  return (2 * static_cast<size_t>(W) * (n + 1) + n) * sizeof(cplx<T>);
}

// launches the compile-time axis kernel of (n, W), if there is one
template <typename T>
bool launch_axis_ct(cplx<T>* data, const cplx<T>* tw, int n, int W, bool strided, int sign, long nlines_or_outer,
                    long S, hipStream_t stream);
// whether n x n planes of elem-byte values have a compile-time kernel (n up to
// 128 in FP32, 100 in FP64)
inline bool plane_ct(int n, size_t elem) { return ct_length(n) && plane_ct_bytes(n, elem) <= kLdsMax; }
// The lengths whose planes are compiled with 256 and with 512 threads, for the
// tuner to choose: the multiples of 16 up to 96.  256 against 512, us for 73 x 64^3
// values: FP32 16 71 / 112, 32 50 / 55, 48 57 / 58, 64 52 / 53, 80 73 / 77, 96 89 /
// 84; FP64 16 118 / 181, 32 99 / 97, 48 100 / 106, 64 200 / 105, 80 211 / 204, 96
// 293 / 212.  The others have one count: up to 32 a stage has at most 256
// butterflies of radix 4 and a block of 512 would idle; above, 512 threads keep
// eight waves on a CU where only one or two planes fit in its LDS.
constexpr bool both_threads(int n) { return n % 16 == 0 && n <= 96; }
// the threads a plane of compiled length n runs with if `threads` are asked for
constexpr int plane_ct_threads(int n, int threads) { return both_threads(n) ? threads : n <= 32 ? 256 : 512; }
// launches it with plane_ct_threads(n, threads), if there is one
template <typename T>
bool launch_plane_ct(cplx<T>* data, const cplx<T>* tw, int n, long planes, int threads, int sign, hipStream_t s);

#ifdef MDFT_FFT_AXIS_CT
template <typename T>
bool launch_axis_ct(cplx<T>* data, const cplx<T>* tw, int n, int W, bool strided, int sign, long nlines_or_outer,
                    long S, hipStream_t stream) {
  bool done = false;
  for_length(n, CtLengths{}, [&](auto nn) {
    constexpr int N = decltype(nn)::value;
    auto go = [&](auto kernel, int w, long nchunk) {
      const long nblk = strided ? nlines_or_outer * nchunk : nchunk;
      throw_if(nblk > 0x7fffffffL, "too many FFT tiles");
      hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(nblk)), dim3(kFftThreads), axis_lds<T>(N, w), stream, data,
                         tw, sign, nlines_or_outer, S, static_cast<unsigned>(nchunk));
      MDFT_HIP_CHECK(hipGetLastError());
      done = true;
    };
    if (!strided) {
      constexpr int w = contiguous_lines<T>(N);
      if (W == w) go(fft_axis_ct_kernel<T, false, N, w>, w, (nlines_or_outer + w - 1) / w);
    } else {
      auto columns = [&](auto ww) {
        constexpr int w = decltype(ww)::value;
        if constexpr (strided_lines(N, w))
          if (W == w) go(fft_axis_ct_kernel<T, true, N, w>, w, (S + w - 1) / w);
      };
      columns(std::integral_constant<int, 4>{});
      columns(std::integral_constant<int, 8>{});
      columns(std::integral_constant<int, 16>{});
      columns(std::integral_constant<int, 32>{});
      columns(std::integral_constant<int, 64>{});
    }
  });
  return done;
}
#endif

}  // namespace mdft
