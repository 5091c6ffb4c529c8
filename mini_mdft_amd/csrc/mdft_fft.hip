// Batched unnormalised 3D c2c FFT for gfx950: mixed-radix Stockham
// transforms of tiles staged in LDS, two launches per 3D transform when a
// (y, z) plane fits in LDS (one pass for z and y together, one for x),
// otherwise one launch per axis.
//
// Replaces the kokkos-fft plans of common/MDFT_Convolution.hpp:198-208 and
// their execution at :328-329 (forward) and :546-547 (backward), both with
// Normalization::none.  A tile holds W lines of length n: for the contiguous
// axis (z) the W lines are W consecutive rows; for the strided axes (y, x) they
// are W neighbouring z columns, so every global access is a run of W (or W*n)
// consecutive complex values.  Each Stockham stage reads one LDS buffer and
// writes the other (radix-4/2/3/5 butterflies, a generic odd-prime DFT up to
// 13), with the twiddles e^{-2 pi i t/n} read from an LDS copy of an FP64
// host table.
//
// Two sets of kernels with the same arithmetic: those here take any length at
// run time; those of mdft_fft_ct.hpp are compiled for each smooth length from 8
// to 128 and serve every axis of such a length and every square plane of one
// that fits in LDS.
#include "mdft_fft.hpp"
#include "mdft_fft_ct.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>

namespace mdft {

namespace {

// One Stockham stage (radix R, Ns = product of the earlier radices) over the
// wvalid lines of a tile: butterfly j of a line reads x[j + r n/R], applies the
// twiddles W_n^{r (j mod Ns) n/(Ns R)}, and writes its outputs at
// (j / Ns) Ns R + (j mod Ns) + r Ns.
template <typename T, int R>
__device__ __forceinline__ void stockham_stage(const cplx<T>* src, cplx<T>* dst, const cplx<T>* tw, int n, int ld,
                                               int Ns, int wvalid, int sign, int tid, int nthreads) {
  const int nb = n / R;
  const int tstep = n / (Ns * R);
  for (int beta = tid; beta < wvalid * nb; beta += nthreads) {
    const int w = beta / nb, j = beta - w * nb;
    const int k = j % Ns;
    const cplx<T>* in = src + w * ld + j;
    cplx<T> v[R];
    v[0] = in[0];
#pragma unroll
    for (int r = 1; r < R; ++r) v[r] = tw_mul<T>(in[r * nb], twiddle<T>(tw, r * k * tstep, sign));
    dft_fixed<T, R>(v, sign, tw, n);
    cplx<T>* out = dst + w * ld + (j / Ns) * Ns * R + k;
#pragma unroll
    for (int r = 0; r < R; ++r) out[r * Ns] = v[r];
  }
}

// The same stage for an odd prime radix 7..13 known only at run time (rare
// lengths): one thread per butterfly output, O(R) LDS reads each, no private
// arrays.
template <typename T>
__device__ __forceinline__ void stockham_stage_generic(const cplx<T>* src, cplx<T>* dst, const cplx<T>* tw, int n,
                                                       int ld, int Ns, int R, int wvalid, int sign, int tid,
                                                       int nthreads) {
  const int nb = n / R;
  const int tstep = n / (Ns * R);
  const int step = n / R;
  for (int it = tid; it < wvalid * nb * R; it += nthreads) {
    const int s = it % R, beta = it / R;
    const int w = beta / nb, j = beta - w * nb;
    const int k = j % Ns;
    const cplx<T>* in = src + w * ld + j;
    cplx<T> acc = in[0];
    for (int r = 1; r < R; ++r) {
      const cplx<T> x = tw_mul<T>(in[r * nb], twiddle<T>(tw, r * k * tstep, sign));
      acc = cfma<T>(acc, x, twiddle<T>(tw, ((r * s) % R) * step, sign));
    }
    dst[w * ld + (j / Ns) * Ns * R + k + s * Ns] = acc;
  }
}

// The same Stockham stage over lines of a 2D LDS tile with a line stride ls
// and an element stride es: element j of line w sits at w ls + j es.  With
// W_FAST, consecutive threads take consecutive lines (the column pass of a
// plane: lines are neighbouring columns, so the accesses of a wave are
// consecutive).
template <typename T, int R, bool W_FAST>
__device__ __forceinline__ void stockham_stage_2d(const cplx<T>* src, cplx<T>* dst, const cplx<T>* tw, int n, int ls,
                                                  int es, int Ns, int nlines, int sign, int tid, int nthreads) {
  const int nb = n / R;
  const int tstep = n / (Ns * R);
  for (int beta = tid; beta < nlines * nb; beta += nthreads) {
    int w, j;
    if (W_FAST) {
      j = beta / nlines;
      w = beta - j * nlines;
    } else {
      w = beta / nb;
      j = beta - w * nb;
    }
    const int k = j % Ns;
    const cplx<T>* in = src + w * ls + j * es;
    cplx<T> v[R];
    v[0] = in[0];
#pragma unroll
    for (int r = 1; r < R; ++r) v[r] = tw_mul<T>(in[r * nb * es], twiddle<T>(tw, r * k * tstep, sign));
    dft_fixed<T, R>(v, sign, tw, n);
    cplx<T>* out = dst + w * ls + ((j / Ns) * Ns * R + k) * es;
#pragma unroll
    for (int r = 0; r < R; ++r) out[r * Ns * es] = v[r];
  }
}

// the stages of one axis over a 2D LDS tile (radices 2, 3, 4, 5), ping-pong
// between a and b; returns the buffer holding the result
template <typename T, bool W_FAST>
__device__ cplx<T>* stockham_2d(cplx<T>* a, cplx<T>* b, const cplx<T>* tw, const FftStages& st, int ls, int es,
                                int nlines, int sign, int tid, int nthreads) {
  int Ns = 1;
  for (int s = 0; s < st.nstages; ++s) {
    const int R = st.radix[s];
    switch (R) {
      case 4: stockham_stage_2d<T, 4, W_FAST>(a, b, tw, st.n, ls, es, Ns, nlines, sign, tid, nthreads); break;
      case 2: stockham_stage_2d<T, 2, W_FAST>(a, b, tw, st.n, ls, es, Ns, nlines, sign, tid, nthreads); break;
      case 3: stockham_stage_2d<T, 3, W_FAST>(a, b, tw, st.n, ls, es, Ns, nlines, sign, tid, nthreads); break;
      default: stockham_stage_2d<T, 5, W_FAST>(a, b, tw, st.n, ls, es, Ns, nlines, sign, tid, nthreads); break;
    }
    __syncthreads();
    cplx<T>* t = a;
    a = b;
    b = t;
    Ns *= R;
  }
  return a;
}

constexpr int kPlaneThreads = 512;

// z and y transforms of one (batch, x) plane of ny x nz contiguous values in
// one pass: the plane is staged in LDS (rows padded to nz + 1), transformed
// along its rows, then along its columns, and written back.  Radices 2-5 only.
template <typename T>
__global__ __launch_bounds__(kPlaneThreads) void fft_plane_kernel(cplx<T>* __restrict__ data, FftStages sz,
                                                                  FftStages sy, const cplx<T>* __restrict__ twz_g,
                                                                  const cplx<T>* __restrict__ twy_g, int sign) {
  extern __shared__ unsigned char lds_raw[];
  const int nz = sz.n, ny = sy.n, ld = nz + 1;
  cplx<T>* bufA = reinterpret_cast<cplx<T>*>(lds_raw);
  cplx<T>* bufB = bufA + ny * ld;
  cplx<T>* twz = bufB + ny * ld;
  cplx<T>* twy = twz + nz;
  const int tid = threadIdx.x;
  const int nth = blockDim.x;
  for (int i = tid; i < nz; i += nth) twz[i] = twz_g[i];
  for (int i = tid; i < ny; i += nth) twy[i] = twy_g[i];
  cplx<T>* plane = data + static_cast<long>(blockIdx.x) * ny * nz;
  for (int t = tid; t < ny * nz; t += nth) {
    const int y = t / nz, z = t - y * nz;
    bufA[y * ld + z] = plane[t];
  }
  __syncthreads();
  cplx<T>* a = stockham_2d<T, false>(bufA, bufB, twz, sz, ld, 1, ny, sign, tid, nth);
  cplx<T>* b = a == bufA ? bufB : bufA;
  a = stockham_2d<T, true>(a, b, twy, sy, 1, ld, nz, sign, tid, nth);
  for (int t = tid; t < ny * nz; t += nth) {
    const int y = t / nz, z = t - y * nz;
    plane[t] = a[y * ld + z];
  }
}

// one fused z/y pass over `planes` planes: the compile-time kernel for square
// planes of the compile-time lengths, else fft_plane_kernel
template <typename T>
void launch_plane(cplx<T>* data, const FftPlan1D& pz, const FftPlan1D& py, long planes, int threads, int sign,
                  hipStream_t s);

bool small_radices(const FftStages& st) {
  for (int s = 0; s < st.nstages; ++s)
    if (st.radix[s] > 5) return false;
  return true;
}

// LDS of the plane kernel: two padded planes and both twiddle tables
template <typename T>
size_t plane_lds(int ny, int nz) {
  return (2 * static_cast<size_t>(ny) * (nz + 1) + ny + nz) * sizeof(cplx<T>);
}
// the fused z/y pass is used untuned when its planes fit in half of the 160 KB
// LDS (at least two blocks of 8 waves per CU); the tuner also tries it up to the
// whole LDS
constexpr size_t kPlaneLdsMax = 80 * 1024;

// One block transforms a tile of W lines of length n.
//   STRIDED = false: line l occupies data[l*n .. l*n+n); the tile is lines
//                    [tile*W, tile*W + W) (clipped at nlines).
//   STRIDED = true : element e of line (o, i) sits at data[(o*n + e)*S + i];
//                    tile = (o, chunk) covers i in [chunk*W, chunk*W + W).
template <typename T, bool STRIDED>
__global__ __launch_bounds__(kFftThreads) void fft_axis_kernel(cplx<T>* __restrict__ data, FftStages st,
                                                               const cplx<T>* __restrict__ tw_g, int sign,
                                                               long nlines_or_outer, long S, int W) {
  extern __shared__ unsigned char lds_raw[];
  const int n = st.n;
  const int ld = n + 1;  // padded row: avoids bank conflicts on column access
  cplx<T>* bufA = reinterpret_cast<cplx<T>*>(lds_raw);
  cplx<T>* bufB = bufA + W * ld;
  cplx<T>* tw = bufB + W * ld;
  const int tid = threadIdx.x;
  for (int i = tid; i < n; i += blockDim.x) tw[i] = tw_g[i];

  long base;
  int wvalid;
  if (!STRIDED) {
    const long l0 = static_cast<long>(blockIdx.x) * W;
    wvalid = static_cast<int>(min(static_cast<long>(W), nlines_or_outer - l0));
    base = l0 * n;
    for (int t = tid; t < wvalid * n; t += blockDim.x) {
      const int w = t / n, e = t - w * n;
      bufA[w * ld + e] = data[base + t];
    }
  } else {
    const long nchunk = (S + W - 1) / W;
    const long o = blockIdx.x / nchunk;
    const long i0 = (blockIdx.x - o * nchunk) * W;
    wvalid = static_cast<int>(min(static_cast<long>(W), S - i0));
    base = o * n * S + i0;
    for (int t = tid; t < wvalid * n; t += blockDim.x) {
      const int e = t / wvalid, w = t - e * wvalid;
      bufA[w * ld + e] = data[base + static_cast<long>(e) * S + w];
    }
  }
  __syncthreads();

  cplx<T>* src = bufA;
  cplx<T>* dst = bufB;
  int Ns = 1;
  for (int s = 0; s < st.nstages; ++s) {
    const int R = st.radix[s];
    switch (R) {
      case 4:
        stockham_stage<T, 4>(src, dst, tw, n, ld, Ns, wvalid, sign, tid, blockDim.x);
        break;
      case 2:
        stockham_stage<T, 2>(src, dst, tw, n, ld, Ns, wvalid, sign, tid, blockDim.x);
        break;
      case 3:
        stockham_stage<T, 3>(src, dst, tw, n, ld, Ns, wvalid, sign, tid, blockDim.x);
        break;
      case 5:
        stockham_stage<T, 5>(src, dst, tw, n, ld, Ns, wvalid, sign, tid, blockDim.x);
        break;
      default:
        stockham_stage_generic<T>(src, dst, tw, n, ld, Ns, R, wvalid, sign, tid, blockDim.x);
        break;
    }
    __syncthreads();
    cplx<T>* t = src;
    src = dst;
    dst = t;
    Ns *= R;
  }

  if (!STRIDED) {
    for (int t = tid; t < wvalid * n; t += blockDim.x) {
      const int w = t / n, e = t - w * n;
      data[base + t] = src[w * ld + e];
    }
  } else {
    for (int t = tid; t < wvalid * n; t += blockDim.x) {
      const int e = t / wvalid, w = t - e * wvalid;
      data[base + static_cast<long>(e) * S + w] = src[w * ld + e];
    }
  }
}

// whether a tile of W columns of stride S has a compiled kernel: it may be wider
// than the stride as long as half of its columns exist (the missing ones are
// computed on for nothing)
bool compiled_columns(int n, int W, long S) { return ct_length(n) && strided_lines(n, W) && 2 * S >= W; }

// default tile: a compiled width where there is one, else about 1024 values.
// Strided axes of compiled lengths: 16 columns, 32 or 64 of short lines; 8 of long
// ones where 16 would leave a CU fewer than 7 tiles (1168 x 128 x 16 FP32 27 us
// against 22, 389 x 96 x 64 27 / 25, but with 8 times the tiles 84 / 104 and
// 82 / 110); no more than it takes for a thin stride.
template <typename T>
int choose_tile_lines(int n, bool strided, long outer, long S) {
  if (strided && ct_length(n)) {
    int W = n <= 16 ? 64 : n <= 32 ? 32 : 16;
    if (n > 64 && outer * ((S + 15) / 16) < 7 * 256) W = 8;
    while (W / 2 >= S && strided_lines(n, W / 2)) W /= 2;
    return W;
  }
  if (!strided && ct_length(n)) return contiguous_lines<T>(n);
  int W = 1024 / n;
  if (W < 1) W = 1;
  if (W > 64) W = 64;
  return W;
}

template <typename T>
void launch_plane(cplx<T>* data, const FftPlan1D& pz, const FftPlan1D& py, long planes, int threads, int sign,
                  hipStream_t s) {
  const int n = pz.st.n;
  const size_t lds = plane_lds<T>(py.st.n, n);
  const dim3 grid(static_cast<unsigned>(planes));
  if (py.st.n != n || !launch_plane_ct<T>(data, pz.twiddles<T>(), n, planes, threads, sign, s)) {
    hipLaunchKernelGGL((fft_plane_kernel<T>), grid, dim3(threads), lds, s, data, pz.st, py.st, pz.twiddles<T>(),
                       py.twiddles<T>(), sign);
  }
  MDFT_HIP_CHECK(hipGetLastError());
}

// W = 0: the default tile.  A strided tile wider than the stride that is not
// compiled is one of the S columns.
template <typename T>
void launch_axis(cplx<T>* data, const FftPlan1D& p, int sign, long nlines_or_outer, long S, bool strided,
                 hipStream_t stream, int W = 0) {
  if (p.st.n == 1 || nlines_or_outer == 0) return;
  if (W <= 0) W = choose_tile_lines<T>(p.st.n, strided, nlines_or_outer, S);
  if (strided && S < W && !compiled_columns(p.st.n, W, S)) W = static_cast<int>(S);
  const size_t lds = axis_lds<T>(p.st.n, W);
  throw_if(lds > kLdsMax, "FFT tile does not fit in LDS");
  const cplx<T>* tw = p.twiddles<T>();
  if (launch_axis_ct<T>(data, tw, p.st.n, W, strided, sign, nlines_or_outer, S, stream)) return;
  if (!strided) {
    const long nblk = (nlines_or_outer + W - 1) / W;
    throw_if(nblk > 0x7fffffffL, "too many FFT tiles");
    hipLaunchKernelGGL((fft_axis_kernel<T, false>), dim3(static_cast<unsigned>(nblk)), dim3(kFftThreads), lds,
                       stream, data, p.st, tw, sign, nlines_or_outer, S, W);
  } else {
    const long nblk = nlines_or_outer * ((S + W - 1) / W);
    throw_if(nblk > 0x7fffffffL, "too many FFT tiles");
    hipLaunchKernelGGL((fft_axis_kernel<T, true>), dim3(static_cast<unsigned>(nblk)), dim3(kFftThreads), lds,
                       stream, data, p.st, tw, sign, nlines_or_outer, S, W);
  }
  MDFT_HIP_CHECK(hipGetLastError());
}

}  // namespace

FftPlan1D::FftPlan1D(int n) {
  throw_if(n <= 0, "FFT length must be positive");
  throw_if(n > 4096, "FFT length above 4096 is not supported");
  st.n = n;
  st.nstages = 0;
  int r = n;
  for (int p : {4, 2, 3, 5, 7, 11, 13}) {
    while (r % p == 0) {
      throw_if(st.nstages >= kFftMaxStages, "too many FFT stages");
      st.radix[st.nstages++] = p;
      r /= p;
    }
  }
  throw_if(r != 1, "FFT length must factor into primes <= 13");
  std::vector<double2> h64(n);
  std::vector<float2> h32(n);
  for (int t = 0; t < n; ++t) {
    const double a = 2.0 * M_PI * static_cast<double>(t) / static_cast<double>(n);
    h64[t].x = std::cos(a);
    h64[t].y = -std::sin(a);
    h32[t].x = static_cast<float>(h64[t].x);
    h32[t].y = static_cast<float>(h64[t].y);
  }
  MDFT_HIP_CHECK(hipMalloc(&tw64_, n * sizeof(double2)));
  MDFT_HIP_CHECK(hipMalloc(&tw32_, n * sizeof(float2)));
  MDFT_HIP_CHECK(hipMemcpy(tw64_, h64.data(), n * sizeof(double2), hipMemcpyHostToDevice));
  MDFT_HIP_CHECK(hipMemcpy(tw32_, h32.data(), n * sizeof(float2), hipMemcpyHostToDevice));
}

FftPlan1D::~FftPlan1D() {
  if (tw64_) (void)hipFree(tw64_);
  if (tw32_) (void)hipFree(tw32_);
}

template <>
const cplx<double>* FftPlan1D::twiddles<double>() const {
  return tw64_;
}
template <>
const cplx<float>* FftPlan1D::twiddles<float>() const {
  return tw32_;
}

Fft3dPlan::Fft3dPlan(int nx_, int ny_, int nz_) : nx(nx_), ny(ny_), nz(nz_), px(nx_), py(ny_), pz(nz_) {}

bool Fft3dPlan::plane_ok(size_t elem) const {
  if (ny == nz && plane_ct(ny, elem)) return true;
  return ny > 1 && nz > 1 && small_radices(py.st) && small_radices(pz.st) &&
         (2 * static_cast<size_t>(ny) * (nz + 1) + ny + nz) * elem <= kLdsMax;
}

template <typename T>
void Fft3dPlan::execute_config(const FftConfig& c, cplx<T>* data, long batch, int sign, hipStream_t stream) const {
  throw_if(sign != -1 && sign != 1, "FFT sign must be -1 or +1");
  const long nxl = nx, nyl = ny, nzl = nz;
  const long planes = batch * nxl;
  if (c.plane) {
    throw_if(!plane_ok(sizeof(cplx<T>)) || planes > 0x7fffffffL ||
                 (c.plane_threads != 256 && c.plane_threads != 512),
             "FFT: the fused plane pass does not apply to this shape");
    // z and y in one pass over each contiguous (y, z) plane
    if (planes > 0) launch_plane<T>(data, pz, py, planes, c.plane_threads, sign, stream);
  } else {
    launch_axis<T>(data, pz, sign, batch * nxl * nyl, 1, false, stream, c.wz);  // z: contiguous lines
    launch_axis<T>(data, py, sign, batch * nxl, nzl, true, stream, c.wy);       // y: stride nz
  }
  launch_axis<T>(data, px, sign, batch, nyl * nzl, true, stream, c.wx);  // x: stride ny*nz
}

template <typename T>
FftConfig Fft3dPlan::default_config() const {
  const bool compiled = ny == nz && plane_ct(ny, sizeof(cplx<T>));
  FftConfig c;
  c.plane = plane_ok(sizeof(cplx<T>)) &&
            (compiled ? plane_ct_bytes(ny, sizeof(cplx<T>)) : plane_lds<T>(ny, nz)) <= kPlaneLdsMax;
  c.plane_threads = compiled ? plane_ct_threads(ny, 512) : 512;
  return c;
}

template <typename T>
void Fft3dPlan::execute(cplx<T>* data, long batch, int sign, hipStream_t stream) const {
  const int k = std::is_same<T, double>::value ? 1 : 0;
  execute_config<T>(tuned_[k] ? cfg_[k] : default_config<T>(), data, batch, sign, stream);
}

// Times the candidate configurations on a scratch array of `batch`
// transforms and keeps the fastest: the tile width of each per-axis pass (the
// compiled ones, else 256, 512, 1024 or 2048 values per tile of the run-time kernel) and, where a (y, z) plane fits in
// LDS, the fused z/y pass with 256 or 512 threads.  Every candidate runs the
// same Stockham stages on the same lines, so the choice changes timing only.
template <typename T>
FftConfig Fft3dPlan::autotune(long batch, hipStream_t s) const {
  const int k = std::is_same<T, double>::value ? 1 : 0;
  if (tuned_[k]) return cfg_[k];
  const long N = static_cast<long>(nx) * ny * nz;
  batch = std::max<long>(1, batch);
  cplx<T>* buf = nullptr;
  MDFT_HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&buf), batch * N * sizeof(cplx<T>)));
  hipEvent_t e0 = nullptr, e1 = nullptr;
  FftConfig best = default_config<T>();
  try {
    MDFT_HIP_CHECK(hipMemsetAsync(buf, 0, batch * N * sizeof(cplx<T>), s));
    MDFT_HIP_CHECK(hipEventCreate(&e0));
    MDFT_HIP_CHECK(hipEventCreate(&e1));
    auto time_ms = [&](auto&& run) {
      run();
      run();
      float best_ms = 1e30f;
      for (int r = 0; r < 3; ++r) {
        MDFT_HIP_CHECK(hipEventRecord(e0, s));
        run();
        MDFT_HIP_CHECK(hipEventRecord(e1, s));
        MDFT_HIP_CHECK(hipEventSynchronize(e1));
        float ms = 0.f;
        MDFT_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
        best_ms = std::min(best_ms, ms);
      }
      return best_ms;
    };
    const long nxl = nx, nyl = ny, nzl = nz;
    // per-axis tile widths: the compiled ones, else tiles of 256 .. 2048 values
    auto candidates = [](int n, long S, bool strided) {
      std::vector<int> w;
      if (!strided && ct_length(n)) w.push_back(contiguous_lines<T>(n));
      if (strided)
        for (int W : {4, 8, 16, 32, 64})
          if (compiled_columns(n, W, S) && (W > 4 || S < 8)) w.push_back(W);
      if (!w.empty()) return w;
      for (int vals : {256, 512, 1024, 2048}) {
        w.push_back(std::max(1, std::min(64, vals / std::max(1, n))));
        if (strided && S < w.back()) w.back() = static_cast<int>(S);
      }
      return w;
    };
    auto best_w = [&](const FftPlan1D& p, long lines, long S, bool strided) {
      int bw = 0;
      float bt = 1e30f;
      for (int W : candidates(p.st.n, S, strided)) {
        if (axis_lds<T>(p.st.n, W) > kLdsMax) continue;
        const float t = time_ms([&] { launch_axis<T>(buf, p, -1, lines, S, strided, s, W); });
        if (t < bt) {
          bt = t;
          bw = W;
        }
      }
      return std::make_pair(bw, bt);
    };
    const auto z = best_w(pz, batch * nxl * nyl, 1, false);
    const auto y = best_w(py, batch * nxl, nzl, true);
    const auto x = best_w(px, batch, nyl * nzl, true);
    FftConfig axes;
    axes.plane = false;
    axes.wz = z.first;
    axes.wy = y.first;
    axes.wx = x.first;
    best = axes;
    float best_t = z.second + y.second + x.second;
    if (plane_ok(sizeof(cplx<T>)) && batch * nxl <= 0x7fffffffL) {
      for (int th : {256, 512}) {
        if (ny == nz && plane_ct(ny, sizeof(cplx<T>)) && plane_ct_threads(ny, th) != th) continue;
        FftConfig c = axes;
        c.plane = true;
        c.plane_threads = th;
        const float t = time_ms([&] {
          launch_plane<T>(buf, pz, py, batch * nxl, th, -1, s);
        }) + x.second;
        if (t < best_t) {
          best_t = t;
          best = c;
        }
      }
    }
  } catch (...) {
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(buf);
    throw;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  MDFT_HIP_CHECK(hipStreamSynchronize(s));
  MDFT_HIP_CHECK(hipFree(buf));
  cfg_[k] = best;
  tuned_[k] = true;
  return best;
}

template void Fft3dPlan::execute<double>(cplx<double>*, long, int, hipStream_t) const;
template void Fft3dPlan::execute<float>(cplx<float>*, long, int, hipStream_t) const;
template void Fft3dPlan::execute_config<double>(const FftConfig&, cplx<double>*, long, int, hipStream_t) const;
template void Fft3dPlan::execute_config<float>(const FftConfig&, cplx<float>*, long, int, hipStream_t) const;
template FftConfig Fft3dPlan::autotune<double>(long, hipStream_t) const;
template FftConfig Fft3dPlan::autotune<float>(long, hipStream_t) const;
template FftConfig Fft3dPlan::default_config<double>() const;
template FftConfig Fft3dPlan::default_config<float>() const;

}  // namespace mdft
