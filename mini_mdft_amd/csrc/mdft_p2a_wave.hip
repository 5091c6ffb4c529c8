// proj2angl of the FP64 and FP32 forms on the compile-time angular grids: a
// block of one wave per mu2 for each (64 consecutive r, theta) (see
// mdft_proj.hip for the sums).
#include "mdft_proj_ct.hpp"
#include "mdft_rows.hpp"

namespace mdft {

namespace {

constexpr int kRows = 64, kXcds = 8;

// the projections of mu2 = B in canonical order: their index, stored channel
// and mup
template <int MMAX, int MRSO, bool CP, int B>
struct MuColumn {
  int count, ip[(MMAX + 1) * (MMAX + 1)], channel[(MMAX + 1) * (MMAX + 1)], mup[(MMAX + 1) * (MMAX + 1)];
  constexpr MuColumn() : count(0), ip(), channel(), mup() {
    const CompactMap<MMAX, MRSO> cm{};
    for (int m = 0, i = 0; m <= MMAX; ++m)
      for (int a = -m; a <= m; ++a)
        for (int mu = 0; mu <= m; mu += MRSO, ++i) {
          if (mu != B * MRSO || (CP && implied_projection(a, mu))) continue;
          ip[count] = i;
          channel[count] = CP ? cm.v[i] : i;
          mup[count++] = a;
        }
  }
};

// wave B: the sums over m of its mu2 for the lane's point (at byte offset of a
// channel) and their phi sums,
//   Z_j = S_0 + sum_{mup > 0} (A cos + i B sin),
//   A = S_mup + S_-mup,  B = S_mup - S_-mup,
// whose cosine and sine parts serve j and nphi - j, into the lane's row of the
// stage: the real part of mu2 = 0 at j npsi, the parts of the others behind it
template <int MMAX, int MRSO, bool CP, int B, typename TP, typename TC, typename F>
__device__ __forceinline__ void p2a_wave(const cplx<TP>* __restrict__ p, long N, unsigned offset, const TabPtrs<TC>& tb,
                                         const TC* __restrict__ w, TC* row, F&& request) {
  using Z = A2pSizes<MMAX, MRSO, 1>;
  constexpr int NPHI = Z::kNphi, NPSI = Z::kNpsi;
  constexpr MuColumn<MMAX, MRSO, CP, B> kCol{};
  // kBatch loads in flight together; left alone, the compiler waits for each
  // where it multiplies it
  constexpr int kBatch = sizeof(TP) == 8 ? 16 : 32;
  TC sr[NPHI], si[NPHI];
#pragma unroll
  for (int a = 0; a < NPHI; ++a) sr[a] = si[a] = TC(0);
#pragma unroll
  for (int c0 = 0; c0 < kCol.count; c0 += kBatch) {
    cplx<TP> v[kBatch];
#pragma unroll
    for (int c = 0; c < kBatch; ++c)
      if (c0 + c < kCol.count)
        v[c] = *reinterpret_cast<const cplx<TP>*>(
            reinterpret_cast<const char*>(p + static_cast<long>(kCol.channel[c0 + c]) * N) + offset);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kBatch; ++c)
      if (c0 + c < kCol.count) {
        const TC wt = w[kCol.ip[c0 + c]];
        const int a = kCol.mup[c0 + c] + MMAX;
        sr[a] = fma(static_cast<TC>(v[c].x), wt, sr[a]);
        si[a] = fma(static_cast<TC>(v[c].y), -wt, si[a]);  // S is the conjugate
      }
  }
  request();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int mup = 1; mup <= MMAX; ++mup) {  // A in place of S_mup, B of S_-mup
    const TC ur = sr[MMAX + mup], ui = si[MMAX + mup], vr = sr[MMAX - mup], vi = si[MMAX - mup];
    sr[MMAX + mup] = ur + vr;
    si[MMAX + mup] = ui + vi;
    sr[MMAX - mup] = ur - vr;
    si[MMAX - mup] = ui - vi;
  }
  const auto put = [&](int j, TC re, TC im) {
    row[j * NPSI + (B > 0 ? 2 * B - 1 : 0)] = re;
    if (B > 0) row[j * NPSI + 2 * B] = im;
  };
#pragma unroll
  for (int j = 0; j <= MMAX; ++j) {
    TC cr = sr[MMAX], ci = si[MMAX], dr = 0, di = 0;  // sum A cos, sum B sin
#pragma unroll
    for (int mup = 1; mup <= MMAX; ++mup) {
      const int t = (mup * j) % NPHI;  // the twiddles of t and nphi - t are conjugate
      const cplx<TC> e = tb.ephi[t > MMAX ? NPHI - t : t];
      const TC sn = t > MMAX ? -e.y : e.y;
      cr = j == 0 ? cr + sr[MMAX + mup] : fma(sr[MMAX + mup], e.x, cr);
      if (B > 0) ci = j == 0 ? ci + si[MMAX + mup] : fma(si[MMAX + mup], e.x, ci);
      if (j > 0) di = fma(si[MMAX - mup], sn, di);
      if (j > 0 && B > 0) dr = fma(sr[MMAX - mup], sn, dr);
    }
    put(j, cr - di, ci + dr);
    if (j > 0) put(NPHI - j, cr + di, ci - dr);
  }
}

// What bounds it is bytes in flight: a single wave with the sums of every mu2
// in its registers (mdft_proj.hip) waits for its projections, then for xi, with
// two waves per SIMD.  Here a wave has one mu2's sums, requests its projections
// 16 (FP64) or 32 at a time and the block's xi before the phi sums, and the
// cosine and sine parts of a phi sum serve two outputs.  A step of the block
// takes whole rows, so that the epilogue has one address per thread.
// Microseconds, one wave against these, fused with get_delta_f: FP64 64^3 mmax
// 5 555 -> 445 (1.7 GB, 351 at the copy rate), 80^3 1052 -> 833, 48^3 mmax 6 569
// -> 474, mmax 3 mrso 1 133 -> 94; FP32 45x36x50 mmax 4 46 -> 38, 48^3 mmax 6 329
// -> 207, 32^3 mmax 5 37 -> 31, 64^3 mmax 5 241 -> 252 (channels a power of two
// apart; 63^3 244 -> 224, 80^3 461 -> 459).  With the xi requested first and 172
// registers FP64 64^3 took 639, held to 168 and 128 registers 804 and 1150.
//
// FUSED: with get_delta_f, if that is known at compile time (FP64 in the full
// order).  Elsewhere it is a branch on xi, behind which the request of xi stays
// in front of the phi sums: FP64 64^3 mmax 5, compact order, 451 us, and 468 where
// the compiler moves it behind them.  In the full order, whose mu2 = 0 has 36
// projections for 21, the early request needs more than 256 registers and leaves
// one wave per SIMD: 640 us against 530, and 506 against 388 for proj2angl alone,
// which requests nothing (FP32 fits either way).
template <int MMAX, int MRSO, typename TP, typename TO, typename TC, bool CP, bool FUSED>
__global__ __launch_bounds__((64 * (MMAX / MRSO + 1))) void proj2angl_mu_kernel(
    const cplx<TP>* __restrict__ p, TO* __restrict__ o, const TO* __restrict__ xi, TO* __restrict__ df,
    const double* __restrict__ wq, long N, long nrb, TabPtrs<TC> tb, double rho0, double* __restrict__ partials,
    double* __restrict__ colpart) {
  using Z = A2pSizes<MMAX, MRSO, 1>;
  constexpr int NPHI = Z::kNphi, NPSI = Z::kNpsi, NMU2 = Z::kNmu2, NJK = NPHI * NPSI, NO = Z::kNo, NTH = Z::kNth;
  const bool fused = sizeof(TC) == 8 && !CP ? FUSED : xi != nullptr;
  using Walk = RowWalk<NJK, 64 * NMU2, kRows>;
  constexpr int kG = Walk::kG, kSteps = Walk::kSteps;
  __shared__ alignas(8) TC stage[kRows * NJK];
  __shared__ double red[NMU2];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the theta blocks of one r range run on the same XCD (block b on XCD b mod
  // 8) and share their projection reads in its L2
  const int q = blockIdx.x / kXcds, th = q % NTH;
  const long rb = static_cast<long>(q / NTH) * kXcds + blockIdx.x % kXcds;
  if (rb >= nrb) return;  // padding block of the XCD ordering
  const long r0 = rb * kRows;
  const int last = static_cast<int>(min(static_cast<long>(kRows) - 1, N - 1 - r0));
  const long base = r0 * NO + th * NJK;
  // thread (sub, col) takes column col of rows sub, sub + kG, ...: the address
  // of a step is a scalar plus a constant of the thread
  const int sub = tid / NJK, col = tid - sub * NJK;
  const bool on = sub < kG;
  // byte offset of the thread's value in step u (Walk::row(sub, u, last))
  const unsigned off0 = on ? (Walk::first(sub, last) * NO + col) * sizeof(TO) : 0;
  const int reach = on ? Walk::reach(sub, last) : 0;
  const auto off = [&](int u) { return off0 + min(u, reach) * static_cast<unsigned>(kG * NO * sizeof(TO)); };
  TO x[kSteps];
  const auto request = [&] {
    if (!fused) return;
    const char* from = reinterpret_cast<const char*>(xi + base);
#pragma unroll
    for (int u = 0; u < kSteps; ++u) x[u] = *reinterpret_cast<const TO*>(from + off(u));
  };
  const double wth = wq[th * NJK];
  cplx<TC> ep[NMU2 * NPSI];  // e^{2 pi i mu2 k/npsi}
#pragma unroll
  for (int i = NPSI; i < NMU2 * NPSI; ++i) ep[i] = tb.epsi[i];
  dispatch_wave<NMU2>(wave, [&](auto bb) {
    p2a_wave<MMAX, MRSO, CP, decltype(bb)::value, TP, TC>(p + r0, N, min(lane, last) * sizeof(cplx<TP>), tb, tb.wts + th * Z::kNp(),
                                                          stage + lane * NJK, request);
  });
  __syncthreads();
  // the c2r over psi, in place: wave w takes j = w, w + nmu2, ... of each row
#pragma unroll
  for (int j0 = 0; j0 < NPHI; j0 += NMU2) {
    const int j = j0 + wave;
    if (j < NPHI) {
      TC* z = stage + lane * NJK + j * NPSI;
      TC v[NPSI], in[NPSI];
#pragma unroll
      for (int k = 0; k < NPSI; ++k) in[k] = z[k];
#pragma unroll
      for (int k = 0; k < NPSI; ++k) {
        v[k] = 0;
#pragma unroll
        for (int b = 1; b < NMU2; ++b) {
          v[k] = fma(in[2 * b - 1], ep[b * NPSI + k].x, v[k]);
          v[k] = fma(-in[2 * b], ep[b * NPSI + k].y, v[k]);
        }
        z[k] = fma(TC(2), v[k], in[0]);
      }
    }
  }
  __syncthreads();
  double acc = 0.0, cs = 0.0, cv = 0.0;
  char* to = reinterpret_cast<char*>((fused ? df : o) + base);
  const auto put = [&](int u) {
    const TO v = static_cast<TO>(stage[(u * kG + sub) * NJK + col]);
    if (!fused) {
      *reinterpret_cast<TO*>(to + off(u)) = v;
    } else {
      const double xv = static_cast<double>(x[u]), vx = static_cast<double>(v);
      const double x2m1 = xv * xv - 1.0;
      acc += vx * wth * x2m1;
      cs += x2m1;
      cv += vx;
      *reinterpret_cast<TO*>(to + off(u)) = static_cast<TO>(2.0 * rho0 * xv * vx);
    }
  };
  if (on) {
    if (last == kRows - 1) {  // no row to leave out before the last step
#pragma unroll
      for (int u = 0; u < kSteps; ++u)
        if ((u + 1) * kG <= kRows || u <= reach) put(u);
    } else {
#pragma unroll
      for (int u = 0; u < kSteps; ++u)
        if (sub <= last && u <= reach) put(u);
    }
  }
  if (colpart != nullptr && fused) {
    // colpart[rb][0][io] = sum_r (xi^2 - 1), colpart[rb][1][io] = sum_r vexc:
    // the threads' sums, then those of a column in the order of sub
    static_assert(2 * kG * sizeof(double) <= kRows * sizeof(TC), "the stage holds the sums");
    double* sums = reinterpret_cast<double*>(stage);
    __syncthreads();  // the stage is read
    if (on) {
      sums[sub * NJK + col] = cs;
      sums[(kG + sub) * NJK + col] = cv;
    }
    __syncthreads();
    if (tid < NJK) {
      double s0 = 0.0, s1 = 0.0;
      for (int g = 0; g < kG; ++g) {
        s0 += sums[g * NJK + tid];
        s1 += sums[(kG + g) * NJK + tid];
      }
      double* cp = colpart + rb * (2 * NO) + th * NJK + tid;
      cp[0] = s0;
      cp[NO] = s1;
    }
  }
  if (fused) {
#pragma unroll
    for (int h = 32; h > 0; h >>= 1) acc += __shfl_xor(acc, h);
    if (lane == 0) red[wave] = acc;
    __syncthreads();
    if (tid == 0) {
      for (int b = 1; b < NMU2; ++b) acc += red[b];
      partials[rb * NTH + th] = acc;
    }
  }
}

}  // namespace

bool proj2angl_mu_waves(const ProjTables& t, bool fp64, long field, bool fused) {
  // Fused FP32 at mmax 5, single wave against these (us): 48^3 97 / 90, 64 x 64 x
  // 32 (2^17) 115.7 / 117.4, 63 x 64^2 219 / 224, 64^3 237 / 250, 96 x 64^2 342 /
  // 347, 80^3 450 / 452, 128 x 64^2 481 / 507: once the chip is full the single
  // wave, which has every channel of its rows in flight, gains on channels that
  // are a power of two apart and loses nowhere.  Alone (63 / 52 at 48^3, 217 /
  // 212 at 64^3), at the other mmax (64^3: mmax 4 159 / 156, mmax 6 782 / 530) and
  // in FP64 the wave per mu2 is as fast or faster.
  return fp64 || !fused || t.mmax != 5 || t.mrso != 2 || field < (1L << 17);
}

template <typename TP, typename TO, typename TC>
bool launch_p2a_wave(const ProjTables& t, long N, const cplx<TP>* p, TO* o, const TO* xi, TO* df,
                     const TabPtrs<TC>& tb, double rho0, double* partials, hipStream_t s, double* colpart, bool compact) {
  bool done = false;
  dispatch_angular(t.mmax, t.mrso, [&](auto mm, auto mr) {
    constexpr int MMAX = decltype(mm)::value, MRSO = decltype(mr)::value;
    const long nrb = (N + kRows - 1) / kRows, blocks = (nrb + kXcds - 1) / kXcds * kXcds * t.ntheta;
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(64 * (MMAX / MRSO + 1)), 0, s, p, o, xi,
                         df, t.w, N, nrb, tb, rho0, partials, colpart);
      MDFT_HIP_CHECK(hipGetLastError());
      done = true;
    };
    if (compact)
      go(proj2angl_mu_kernel<MMAX, MRSO, TP, TO, TC, true, true>);
    else if (sizeof(TC) == 4 || xi != nullptr)
      go(proj2angl_mu_kernel<MMAX, MRSO, TP, TO, TC, false, true>);
    else
      go(proj2angl_mu_kernel<MMAX, MRSO, TP, TO, TC, false, sizeof(TC) == 4>);
  });
  return done;
}

template bool launch_p2a_wave<double, double, double>(const ProjTables&, long, const cplx<double>*, double*,
                                                      const double*, double*, const TabPtrs<double>&, double, double*,
                                                      hipStream_t, double*, bool);
template bool launch_p2a_wave<float, float, float>(const ProjTables&, long, const cplx<float>*, float*, const float*,
                                                   float*, const TabPtrs<float>&, double, double*, hipStream_t, double*,
                                                   bool);

}  // namespace mdft
