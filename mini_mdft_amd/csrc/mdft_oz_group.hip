// The per-(q, -q) pass of Convolution::execute (common/MDFT_Convolution.hpp:
// 376-543: rotation to the q frame, c(|q|) interpolation, OZ product, chop,
// inverse rotation, stores) over groups of consecutive stars, on the matrix
// cores.
//
// A star is the set of q = (+-kx, +-ky, +-kz): up to four (q, -q) pairs, eight
// vectors of np projections, which share |q| (the c(q) row and its lerp
// weights) and theta_q (the real rotation matrices d^l).  Both rotations and
// the OZ product are then products of a matrix of the star with 16 columns
// (8 vectors x re, im): one 16-wide MFMA tile.
//   rotation  D(m, chi, mu2) = sum_mup G(m, mup, mu2) d^m_{mup,chi}: K = 2m+1
//             (padded to a multiple of 4 with zeros of d); the -q vectors take
//             d_{mup,-chi} (-1)^m, i.e. the mirrored output row;
//   OZ        gamma(m, mu2) = sum_(n, nu2) c D(n, chi, |nu2|) for each chi, a
//             complex product: K = terms x (Cr, Ci), four terms per step;
//   inverse   out(m, mup, mu2) = sum_chi gamma d_{mup,chi}; the -q vectors use
//             sum_chi gamma d_{mup,-chi} = (-1)^mup sum_chi (-1)^chi gamma d_{-mup,chi}.
// The data are the A operand (rows = 16 columns of the star) and d or c the B
// operand, so that a lane of the result holds the four consecutive values (q
// re, im, -q re, im) of one pair and writes them with one or two wide stores.
// v_mfma_f32_16x16x4_f32 accumulates its four products as sequential FMAs in
// the order of K: the sums run in the order of the one-output-per-thread
// kernels, bit for bit where c is real (ten grids of 600 to 36 000 stars with
// both kernels, in both channel orders).
//
// What bounds the pass.  Per star it moves 2 x 8 x np values and does 209
// kflop at mmax 5, 140 MFMA tiles: 4480 cycles of a SIMD, 70 us for the
// 35 937 stars of 64^3.  The one-block-per-star kernel takes 334 us there, and
// still 232 us with its gathers, c(q) loads, rotations and most of its OZ
// product taken out: what is left is block launches, a chain of dependent loads
// (star, pair record, gathers), seven barriers, and gathers that touch a
// 64-byte segment per 8 bytes.  So here:
//   * a block of 8 waves takes 8 consecutive stars, whose points are runs of 8
//     consecutive z: the loads and stores of a channel are 64-byte segments,
//     spread over all the block's lanes;
//   * every index is computed from the star index; the block is persistent and
//     requests the next group's projections, c(q) rows and d table into
//     registers while it computes the current one;
//   * each star belongs to one wave, so that the three products need no
//     barrier between them; a wave requests all operands of a step before its
//     first product.
// 64^3, mmax 5: 334 -> 217 us (80^3: 576 -> 399, 96^3: 961 -> 685 to 705); two waves
// per SIMD (LDS holds 8 stars of 19 KB) leave the OZ product at about half of
// the matrix rate.  Measured and left out: 4-wave blocks of 4 stars, two per CU
// (276 us), two waves per star (spills at 128 registers: 424 us), and FP64 (4
// stars of two waves each: 454 against 508 us at 64^3, but 870 against 847 at
// 80^3 and 208 against 189 at 48^3).
#include "mdft_oz_group.hpp"

#include <hip/hip_ext.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "mdft_proj.hpp"

namespace mdft {

namespace {

constexpr int kStars = 8, kWaves = kStars, kThreads = 64 * kWaves;  // a wave per star
constexpr int kXcds = 8;
constexpr size_t kLdsMax = 160 * 1024;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

struct alignas(16) OzStarMeta {
  int iq;
  float al, bl;
};

// Compile-time shape of an angular grid.  Terms tau = (n, nu2), n ascending,
// nu2 = -n/mrso .. n/mrso; outputs o = (m, mu2), m ascending.
template <int MMAX, int MRSO>
struct Sh {
  static constexpr int W = 2 * MMAX + 1;
  static constexpr int km(int m) { return m / MRSO + 1; }
  static constexpr int tau0(int n) {  // terms of the n' < n
    int a = 0;
    for (int k = 0; k < n; ++k) a += 2 * (k / MRSO) + 1;
    return a;
  }
  static constexpr int ofs(int m) {  // outputs of the m' < m
    int a = 0;
    for (int k = 0; k < m; ++k) a += km(k);
    return a;
  }
  static constexpr int rows(int m) {  // projections of the m' < m
    int a = 0;
    for (int k = 0; k < m; ++k) a += (2 * k + 1) * km(k);
    return a;
  }
  static constexpr int NT = tau0(MMAX + 1), NO = ofs(MMAX + 1), NP = rows(MMAX + 1);
  static constexpr int NG = (NT + 3) / 4;  // steps of four terms at chi = 0
  static constexpr int abs(int x) { return x < 0 ? -x : x; }
  static constexpr int nout(int chi) { return NO - ofs(abs(chi)); }
  static constexpr int nins(int chi) { return NT - tau0(abs(chi)); }
  // c rows: the (chi, m, mu2) rows of terms, each padded to an odd length (the
  // 16 rows of a step start 2 banks apart mod 32 at worst)
  static constexpr int ldc(int chi) { return nins(chi) | 1; }
  static constexpr int cofs(int chi) {
    int a = 0;
    for (int x = -MMAX; x < chi; ++x) a += nout(x) * ldc(x);
    return a;
  }
  static constexpr int terms() {
    int a = 0;
    for (int x = -MMAX; x <= MMAX; ++x) a += nout(x) * nins(x);
    return a;
  }
  static constexpr int NC = cofs(MMAX + 1);
  static constexpr int NCP = (NC + 1) & ~1;  // a row is a whole number of 16-byte loads
  // LDS rows of 16 values of one star, one block of 2m+1 rows per (m, mu2).
  // Steps with terms of n < |chi| read up to PADF rows before the first block,
  // and the K padding of the last block reads up to three rows past it.  The
  // four terms of an OZ step read the middle rows of their blocks + chi, and a
  // row covers 16 of the 64 banks: each block is placed so that its middle
  // row's number mod 4 differs from those of the blocks it shares a step with.
  static constexpr int PADF = MMAX < 2 ? MMAX : 2;
  static constexpr bool share_step(int m, int u, int m2, int u2) {
    for (int a = -1; a <= 1; a += 2)
      for (int b = -1; b <= 1; b += 2)
        if ((tau0(m) + m / MRSO + a * u) / 4 == (tau0(m2) + m2 / MRSO + b * u2) / 4) return true;
    return false;
  }
  struct Rows {
    int v[NO] = {};
    constexpr Rows() {
      int bm[NO] = {}, bu[NO] = {}, a = PADF, i = 0;
      for (int k = 0; k <= MMAX; ++k)
        for (int u = 0; u < km(k); ++u, ++i) {
          int p = 0;
          for (; p < 4; ++p) {
            bool ok = true;
            for (int x = 0; x < i; ++x)
              if (share_step(k, u, bm[x], bu[x]) && (v[x] + bm[x]) % 4 == (a + p + k) % 4) ok = false;
            if (ok) break;
          }
          a += p % 4;
          v[i] = a;
          bm[i] = k;
          bu[i] = u;
          a += 2 * k + 1;
        }
    }
  };
  __host__ __device__ static constexpr int rowbase(int m, int mu2) {
    constexpr Rows r{};
    return r.v[ofs(m) + mu2];
  }
  static constexpr int NROW = rowbase(MMAX, km(MMAX) - 1) + 2 * MMAX + 1 + 3;
  // d^m blocks, m >= 1: K4(m) rows (mup + m) of CW columns (chi + m)
  static constexpr int k4(int m) { return (2 * m + 1 + 3) / 4 * 4; }
  static constexpr int CW = k4(MMAX);
  static constexpr int dofs(int m) {
    int a = 0;
    for (int k = 1; k < m; ++k) a += k4(k) * CW;
    return a;
  }
  static constexpr int ND = dofs(MMAX + 1);
  static constexpr int NE = (MMAX + 1) * (MMAX + 2) / 2 * W;  // entries of a half d table
};

template <int MMAX, int MRSO>
struct Lay {
  using S = Sh<MMAX, MRSO>;
  static constexpr size_t r16(size_t b) { return (b + 15) / 16 * 16; }
  // one star: rows | c terms | d (and what the last d rows' padding lanes reach past it)
  static constexpr size_t xb = S::NROW * 16 * sizeof(float);
  static constexpr size_t cb = r16(S::NCP * 2 * sizeof(float));
  static constexpr size_t db = r16((S::ND + (16 - S::CW) * S::CW + 16) * sizeof(float));
  // an odd number of 8-value units: the stars' rows start 8 banks apart
  static constexpr size_t region = (xb + cb + db + 8 * sizeof(float) - 1) / (8 * sizeof(float)) * (8 * sizeof(float)) +
                                   ((xb + cb + db + 8 * sizeof(float) - 1) / (8 * sizeof(float)) % 2 ? 0 : 8 * sizeof(float));
  // all stars, and two buffers of the phases e^{-i mup phi} of their four pairs
  static constexpr size_t total = kStars * region + r16(2 * kStars * 4 * S::W * 2 * sizeof(float));
  static constexpr int per_cu = static_cast<int>(kLdsMax / total);
  static_assert(S::NO <= 16 && total <= kLdsMax, "a group's LDS");
};

struct GroupArgs {
  float2* p;
  const float* dtab;
  const float2* ctab;
  const OzStarMeta* meta;
  const float2* phase;
  const int* dcode;
  const int* chrec;
  int nx, ny, nz, hy, hz, nbatch;
  int nstars, ngroups, chunk;
  long N, pstride;
  float chop_eps;
};

// channel records: LDS row | row of (m, -mup, mu2) << 10 | mup + mmax << 20 | flags
constexpr int kRecOdd = 1 << 24, kRecFold = 1 << 25;
// places of a half d table's entry: place | mirror << 12 | flags
constexpr int kPlaceNeg = 1 << 24, kPlaceValid = 1 << 25;

// order LDS accesses of the lanes of one wave
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// products in one fixed rounding (the compiler's choice of which product to
// fuse depends on the code around it): x e^{i phi} with e = (ex, ey), and the
// lerp of two c rows, as the one-output-per-thread kernels compile to
__device__ __forceinline__ float2 turn(float2 x, float ex, float ey) {
  return make_float2(fma(x.x, ex, -(x.y * ey)), fma(x.y, ex, x.x * ey));
}
// where a lane's vector of its star lies: the own point, and what the store
// rules need
struct Point {
  int at;
  bool store, self, singular;
};

template <typename A>
__device__ __forceinline__ Point point_of(const A& a, int star, int j, int side) {
  const int s = min(star, a.nstars - 1);
  const int r = s / a.hz, az = s - r * a.hz, ax = r / a.hy, ay = r - ax * a.hy;
  const bool okx = !(j & 1) || (ax != 0 && 2 * ax != a.nx), oky = !(j & 2) || (ay != 0 && 2 * ay != a.ny);
  const int x = (j & 1) && okx ? a.nx - ax : ax, y = (j & 2) && oky ? a.ny - ay : ay;
  const int xm = x == 0 ? 0 : a.nx - x, ym = y == 0 ? 0 : a.ny - y, zm = az == 0 ? 0 : a.nz - az;
  // in the self-conjugate z planes q is the member the reference's sweep meets first
  const bool q = zm != az || y < ym || (y == ym && x <= xm);
  Point t;
  t.self = xm == x && ym == y && zm == az;
  t.singular = t.self && (x == a.nx / 2 || y == a.ny / 2 || az == a.nz / 2);
  // at a self-conjugate point the -q store is the one that stays
  t.store = star < a.nstars && okx && oky && q && (side == 1 || !t.self);
  t.at = side ? (xm * a.ny + ym) * a.nz + zm : (x * a.ny + y) * a.nz + az;
  return t;
}

// v with its sign flipped where mask is kSign (0: v)
constexpr unsigned kSign = 0x80000000u;
__device__ __forceinline__ float flip(float v, unsigned mask) {
  return __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) ^ mask);
}
__device__ __forceinline__ unsigned sign_if(bool neg) { return neg ? kSign : 0u; }

template <int MMAX, int MRSO, bool CP>
__global__ __launch_bounds__(kThreads) void oz_group_kernel(GroupArgs a) {
  using S = Sh<MMAX, MRSO>;
  using L = Lay<MMAX, MRSO>;
  constexpr int NCH = CP ? compact_count<MMAX, MRSO>() : S::NP;
  constexpr int NI = (NCH + kWaves - 1) / kWaves;  // channels per wave
  constexpr int NCV = S::NCP / 2;                  // 16-byte pieces of a c row
  constexpr int NCI = (NCV + 63) / 64, NDI = (S::NE + 63) / 64;  // of them, and of half d entries, per lane
  constexpr int W = S::W, NPH = kStars * 4 * W;    // phases of a group
  static_assert(NPH <= kThreads, "one phase per thread");
  extern __shared__ __align__(16) unsigned char lds_raw[];
  float2* ph = reinterpret_cast<float2*>(lds_raw + kStars * L::region);  // [2][Z][4][W]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // load / store lanes: star t, vector v = 2 j + side; a wave covers a channel
  const int t = lane & 7, v = lane >> 3, side = v & 1, j = v >> 1;
  // the byte offset of this vector's column in its star's rows
  int xtoff = t * static_cast<int>(L::region) + 2 * v * static_cast<int>(sizeof(float));

  // the wave's star (star `wave` of the group): rows, c terms, d blocks
  float* X = reinterpret_cast<float*>(lds_raw + wave * L::region);
  float* C = reinterpret_cast<float*>(lds_raw + wave * L::region + L::xb);
  float* D = reinterpret_cast<float*>(lds_raw + wave * L::region + L::xb + L::cb);
  // MFMA lanes: data column (A row) or result column col, K index and result
  // group kq (the lane's four results: data columns 4 kq + r)
  const int col = lane & 15, kq = lane >> 4;

  // OZ lanes: per step g the term tau = 4 g + kq: where its two operands (the
  // lane's component and the other one) are at chi = 0, and their signs:
  // re: cr xr -+ ci xi, im: +-cr xi + ci xr (upper signs: plain, lower:
  // conjugate).  Rows of -q vectors are held mirrored (chi at -chi)
  int aoff[S::NG], adir[S::NG];
  unsigned as1[S::NG], as2[S::NG];
  const int cpart = col & 1, cv = col >> 1;
#pragma unroll
  for (int g = 0; g < S::NG; ++g) {
    const int tau = min(4 * g + kq, S::NT - 1);
    int off = 0;
    bool cj = false;
    int k = 0;
#pragma unroll
    for (int n = 0; n <= MMAX; ++n)
#pragma unroll
      for (int nu2 = -(n / MRSO); nu2 <= n / MRSO; ++nu2, ++k)
        if (tau == k) {
          off = S::rowbase(n, nu2 < 0 ? -nu2 : nu2) + n;
          cj = nu2 >= 0;
        }
    const int vec = cv ^ (cj ? 1 : 0);
    aoff[g] = off * 16 + 2 * vec + cpart;
    adir[g] = (vec & 1) ? -16 : 16;
    as1[g] = sign_if(cpart && cj);
    as2[g] = sign_if(!cpart && !cj);
  }
  const int other = cpart ? -1 : 1;
  // the lane's output (m, mu2): its row at chi = 0
  int orow = 0;
  {
    int k = 0;
#pragma unroll
    for (int m = 0; m <= MMAX; ++m)
#pragma unroll
      for (int mu2 = 0; mu2 < S::km(m); ++mu2, ++k)
        if (col == k) orow = S::rowbase(m, mu2) + m;
  }
  orow = orow * 16 + 4 * kq;
  // the lane's first c term at |chi|
  int coff[MMAX + 1];
#pragma unroll
  for (int ac = 0; ac <= MMAX; ++ac)
    coff[ac] = 2 * (min(max(col - S::ofs(ac), 0), S::nout(ac) - 1) * S::ldc(ac) + kq - S::tau0(ac));

  // the block's items: XCD x runs a contiguous range of groups, the fields of a batch innermost
  const int xcd = blockIdx.x % kXcds, nslots = gridDim.x / kXcds, nitems = a.chunk * a.nbatch;
  struct Item {
    int rest, group, job;
    bool live;
  };
  auto item = [&](int r) {
    Item it;
    it.rest = r;
    it.group = xcd * a.chunk + (a.nbatch == 1 ? r : static_cast<int>(static_cast<unsigned>(r) / a.nbatch));
    it.job = a.nbatch == 1 ? 0 : static_cast<int>(static_cast<unsigned>(r) % a.nbatch);
    it.live = r < nitems && it.group < a.ngroups;
    return it;
  };
  Item cur = item(blockIdx.x / kXcds);
  if (!cur.live) return;

  for (int i = tid; i < static_cast<int>(L::total / 16); i += kThreads)
    reinterpret_cast<f32x4*>(lds_raw)[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  int rec[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) rec[i] = a.chrec[min(i * kWaves + wave, NCH - 1)];
  int dplace[NDI];
#pragma unroll
  for (int k = 0; k < NDI; ++k) {
    const int e = lane + k * 64;
    dplace[k] = e < S::NE ? a.dcode[e] : 0;
  }
  // the phase this thread keeps in ph: star, pair, mup, and the signs of its
  // pair: phi of (-kx, ky) is pi - phi, of (kx, -ky) -phi
  const int pe = min(tid, NPH - 1), pstar = pe / (4 * W), pmup = pe % W - MMAX;
  const int pam = pmup < 0 ? -pmup : pmup, pj = pe / W % 4;
  const unsigned psx = sign_if((pj & 1) && (pam & 1));
  const unsigned psy = sign_if((((pj & 1) && !(pam & 1)) != ((pj & 2) != 0)) != (pmup < 0));

  float2 xr[NI];
  f32x4 lo[NCI], hi[NCI];
  float dr[NDI];
  float2 phr = make_float2(0.f, 0.f);
  Point pt, ptn;
  OzStarMeta mt, mtn;
  auto star_meta = [&](const Item& it) { return a.meta[min(it.group * kStars + wave, a.nstars - 1)]; };
  const long cstep = a.pstride * kWaves;  // from one of the wave's channels to its next

  // requests an item's projections, d table and phase (long before their use:
  // HBM), and its c(q) rows (L2; after the OZ product, whose operands need the registers)
  const float2* src = nullptr;
  unsigned soff = 0;
  auto request_x = [&](int i0, int i1) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (i >= i0 && i < i1 && (i + 1 < NI || i * kWaves + wave < NCH)) xr[i] = (src + i * cstep)[soff];
  };
  auto request = [&](const Item& it, Point& pnt) {
    pnt = point_of(a, it.group * kStars + t, j, side);
    src = a.p + it.job * a.N + wave * a.pstride;
    soff = static_cast<unsigned>(pnt.at);
    const float* drow = a.dtab + static_cast<long>(min(it.group * kStars + wave, a.nstars - 1)) * S::NE;
#pragma unroll
    for (int k = 0; k < NDI; ++k) dr[k] = drow[min(lane + k * 64, S::NE - 1)];
    phr = a.phase[static_cast<long>(min(it.group * kStars + pstar, a.nstars - 1)) * (MMAX + 1) + pam];
  };
  auto request_c = [&](const OzStarMeta& m) {
    const f32x4* crow = reinterpret_cast<const f32x4*>(a.ctab) + static_cast<long>(m.iq) * NCV;
#pragma unroll
    for (int k = 0; k < NCI; ++k) {
      const int q = min(lane + k * 64, NCV - 1);
      lo[k] = crow[q];
      hi[k] = crow[q + NCV];
    }
  };
  auto keep_phase = [&](int b) {
    if (tid < NPH) ph[b * NPH + tid] = make_float2(flip(phr.x, psx), flip(phr.y, psy));
  };

  // The rotations of the wave's blocks (m, mu2), m >= 1 (d^0 = 1).  To the q
  // frame (:427-443): the -q vectors' rows come out mirrored, times (-1)^m.
  // Back (:518-541): the -q rows come out mirrored, times (-1)^{m + mup}.  All
  // operands are requested before the first product.
  auto rotate = [&](auto backc) {
    constexpr bool BACK = decltype(backc)::value;
    constexpr int KS = S::CW / 4;
    float b[MMAX + 1][KS], x[S::NO][KS];
    const unsigned odd = sign_if(col & 1);
    int blk = 0;
#pragma unroll
    for (int m = 1; m <= MMAX; ++m) {
#pragma unroll
      for (int s = 0; s < KS; ++s)
        if (s < S::k4(m) / 4)
          b[m][s] = BACK ? D[S::dofs(m) + col * S::CW + 4 * s + kq] : D[S::dofs(m) + (4 * s + kq) * S::CW + col];
#pragma unroll
      for (int mu2 = 0; mu2 < S::km(m); ++mu2, ++blk)
#pragma unroll
        for (int s = 0; s < KS; ++s)
          if (s < S::k4(m) / 4) x[blk][s] = X[(S::rowbase(m, mu2) + 4 * s + kq) * 16 + col];
    }
    __builtin_amdgcn_sched_barrier(0);
    blk = 0;
#pragma unroll
    for (int m = 1; m <= MMAX; ++m)
#pragma unroll
      for (int mu2 = 0; mu2 < S::km(m); ++mu2, ++blk) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; ++s)
          if (s < S::k4(m) / 4) acc = mfma4(x[blk][s], b[m][s], acc);
#pragma unroll
        for (int r = 2; r < 4; ++r) acc[r] = BACK ? flip(acc[r], odd) : ((m & 1) ? -acc[r] : acc[r]);
        if (col <= 2 * m) *reinterpret_cast<f32x4*>(&X[(S::rowbase(m, mu2) + col) * 16 + 4 * kq]) = acc;
      }
  };

  // OZ product (:468-496) and chop (:514-517) of every |chi|.  chi and
  // -chi share their rows (the -q vectors' are mirrored), so both are read
  // before either is written; gamma is written unmirrored, the -q vectors'
  // times (-1)^chi
  auto oz_all = [&]() {
    struct Ops {
      float a1[S::NG], a2[S::NG];
      f32x2 c[S::NG];
    };
    auto load = [&](auto chic, Ops& o) {
      constexpr int chi = decltype(chic)::value, ac = chi < 0 ? -chi : chi;
      constexpr int tau0 = S::tau0(ac);
      const float* c = C + 2 * S::cofs(chi) + coff[ac];
#pragma unroll
      for (int g = tau0 / 4; g < S::NG; ++g) {
        const float* xp = X + (aoff[g] + chi * adir[g]);
        o.a1[g] = xp[0];
        o.a2[g] = xp[other];
        o.c[g] = *reinterpret_cast<const f32x2*>(&c[8 * g]);
      }
    };
    auto product = [&](auto chic, const Ops& o) {
      constexpr int chi = decltype(chic)::value, ac = chi < 0 ? -chi : chi;
      constexpr int tau0 = S::tau0(ac);
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int g = tau0 / 4; g < S::NG; ++g) {
        f32x2 cc = o.c[g];
        if (4 * g < tau0 || 4 * g + 3 >= S::NT) {  // a step with terms of n < |chi|, or past the last
          const bool in = 4 * g + kq >= tau0 && 4 * g + kq < S::NT;
          cc[0] = in ? cc[0] : 0.f;
          cc[1] = in ? cc[1] : 0.f;
        }
        acc = mfma4(flip(o.a1[g], as1[g]), cc[0], acc);
        acc = mfma4(flip(o.a2[g], as2[g]), cc[1], acc);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[r] = fabs(acc[r]) < a.chop_eps ? 0.f : ((chi & 1) && r >= 2 ? -acc[r] : acc[r]);
      return acc;
    };
    auto write = [&](auto chic, const f32x4& acc) {
      constexpr int chi = decltype(chic)::value, ac = chi < 0 ? -chi : chi;
      if (col >= S::ofs(ac) && col < S::NO) *reinterpret_cast<f32x4*>(&X[orow + chi * 16]) = acc;
    };
    auto both = [&](auto acc_, const Ops& u, const Ops& w) {
      constexpr int A = decltype(acc_)::value;
      const f32x4 r0 = product(std::integral_constant<int, A>{}, u);
      if constexpr (A > 0) {
        const f32x4 r1 = product(std::integral_constant<int, -A>{}, w);
        write(std::integral_constant<int, -A>{}, r1);
      }
      write(std::integral_constant<int, A>{}, r0);
    };
    // the operands of the next |chi| are requested before the products of the
    // current one (their rows are others): the eight waves run in step, and
    // LDS would idle in their products and the matrix cores in their loads
    auto all = [&](auto self, auto acc_, Ops& u, Ops& w) {
      constexpr int A = decltype(acc_)::value;
      // a part of the next item's projections at a time: requested at once
      // after a barrier they would queue up in front of the products
      request_x(A * NI / (MMAX + 1), (A + 1) * NI / (MMAX + 1));
      if constexpr (A < MMAX) {
        Ops un, wn;
        load(std::integral_constant<int, A + 1>{}, un);
        load(std::integral_constant<int, -A - 1>{}, wn);
        __builtin_amdgcn_sched_barrier(0);
        both(acc_, u, w);
        __builtin_amdgcn_sched_barrier(0);
        self(self, std::integral_constant<int, A + 1>{}, un, wn);
      } else {
        both(acc_, u, w);
      }
    };
    Ops u, w;
    load(std::integral_constant<int, 0>{}, u);
    all(all, std::integral_constant<int, 0>{}, u, w);
  };

  mt = star_meta(cur);
  request(cur, pt);
  request_x(0, NI);
  request_c(mt);
  __syncthreads();  // the zeros are in place
  keep_phase(0);
  int buf = 0;

  while (true) {
    // past the last item the current one is requested again: unconditional
    // requests let the registers of this item's inputs end with their use
    Item next = item(cur.rest + nslots);
    const bool more = next.live;
    if (!more) next = cur;
    // opaque once per trip: the addresses formed from these are cheap, and
    // kept across trips they would take every register the operands need
    asm volatile("" : "+v"(xtoff));
#pragma unroll
    for (int g = 0; g < S::NG; ++g) asm volatile("" : "+v"(adir[g]));
    float* xt = reinterpret_cast<float*>(lds_raw + xtoff);
    mtn = star_meta(next);
    __syncthreads();  // the rows, c and d of the previous item are free; its phases are in place
    const float2* pl = ph + buf * NPH + (t * 4 + j) * W;  // e^{-i mup phi} of this lane's pair

    // projections into the rows, phased; an implied projection from its partner
    {
      float* xm = xt + (side ? -2 : 2);  // the vector at the mirrored point
      float2 e[NI];  // all LDS reads before the first write
#pragma unroll
      for (int i = 0; i < NI; ++i) e[i] = pl[(rec[i] >> 20) & 15];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if (i + 1 < NI || i * kWaves + wave < NCH) {
          const int r = rec[i], row = (r & 1023) * 16, frow = ((r >> 10) & 1023) * 16;
          const unsigned odd = (r & kRecOdd) ? kSign : 0u;
          const float2 z = turn(xr[i], e[i].x, e[i].y);
          *reinterpret_cast<f32x2*>(&xt[row]) = f32x2{z.x, z.y};
          if (CP && (r & kRecFold))
            *reinterpret_cast<f32x2*>(&xm[frow]) = f32x2{flip(z.x, odd), flip(z.y, odd ^ kSign)};
        }
      }
    }
    // the lerped c row and the mirrored d blocks of the wave's star
    {
      const float al = mt.al, bl = mt.bl;
#pragma unroll
      for (int k = 0; k < NCI; ++k) {
        const int q = lane + k * 64;
        f32x4 w;
#pragma unroll
        for (int u = 0; u < 4; ++u) w[u] = fma(al, hi[k][u], bl * lo[k][u]);
        if (k + 1 < NCI || q < NCV) reinterpret_cast<f32x4*>(C)[q] = w;
      }
#pragma unroll
      for (int k = 0; k < NDI; ++k) {
        const int c = dplace[k];
        if (c & kPlaceValid) {
          D[c & 0xfff] = dr[k];
          D[(c >> 12) & 0xfff] = flip(dr[k], (c & kPlaceNeg) ? kSign : 0u);
        }
      }
    }
    __syncthreads();
    request(next, ptn);

    rotate(std::false_type{});
    wave_sync();
    oz_all();
    wave_sync();
    rotate(std::true_type{});
    request_c(mtn);
    keep_phase(buf ^ 1);
    __syncthreads();

    // the rows, unphased, to q and -q; a partner channel takes the pair's
    // combination g_+ + (-1)^mup conj(g_- at the mirrored point)
    {
      float2* dst = a.p + cur.job * a.N + wave * a.pstride;
      const unsigned off = static_cast<unsigned>(pt.at);
      // the implied projection's vector at the mirrored point (rows of -q
      // vectors are mirrored: its row of -mup is the row of +mup)
      const bool mside = pt.self ? side : !side;
      const float* xm = xt + (pt.self ? 0 : side ? -2 : 2);
      const unsigned sg = sign_if(pt.singular);
#pragma unroll
      for (int i = 0; i < NI; ++i, dst += cstep) {
        if (i + 1 < NI || i * kWaves + wave < NCH) {
          const int r = rec[i], rp = (r & 1023) * 16, rm = ((r >> 10) & 1023) * 16;
          const int row = side ? rm : rp, frow = mside ? rp : rm;
          const unsigned odd = (r & kRecOdd) ? kSign : 0u;
          const float2 e = pl[(r >> 20) & 15];
          const f32x2 x = *reinterpret_cast<const f32x2*>(&xt[row]);
          float2 z = turn(make_float2(x[0], x[1]), e.x, -e.y);
          z.y = flip(z.y, sg);
          if (CP && (r & kRecFold)) {
            const f32x2 g = *reinterpret_cast<const f32x2*>(&xm[frow]);
            const float2 h = turn(make_float2(g[0], g[1]), e.x, e.y);
            z.x += flip(h.x, odd);
            z.y += flip(h.y, sg ^ odd ^ kSign);
          }
          if (pt.store) dst[off] = z;
        }
      }
    }
    if (!more) break;
    cur = next;
    mt = mtn;
    pt = ptn;
    buf ^= 1;
  }
}

// e^{i mup phi} of q = (q0, q1) as phase_pow of mdft_conv.hip; c(q) row and
// weights as oz_meta_kernel there
__global__ __launch_bounds__(256) void star_meta_kernel(OzStarMeta* __restrict__ meta, float2* __restrict__ phase,
                                                        const double* __restrict__ k, int nx, int ny, int hy, int hz,
                                                        long nstars, int mmax, int nq, double dq) {
  const long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= nstars) return;
  const int az = static_cast<int>(i % hz);
  const long r = i / hz;
  const int ay = static_cast<int>(r % hy), ax = static_cast<int>(r / hy);
  const double q0 = k[ax], q1 = k[nx + ay], q2 = k[nx + ny + az];
  const double qn = sqrt(q0 * q0 + q1 * q1 + q2 * q2);
  const double eff = qn / dq;
  int iq = static_cast<int>(eff);
  const double alpha = eff - static_cast<double>(iq);
  if (iq > nq - 2) iq = nq - 2;  // unreachable for |q| <= qmax (nq has 1.5 rows of margin)
  OzStarMeta m;
  m.iq = iq;
  m.al = static_cast<float>(alpha);
  m.bl = static_cast<float>(1.0 - alpha);
  meta[i] = m;
  const double rxy = sqrt(q0 * q0 + q1 * q1);
  const double c1 = rxy > 0.0 ? q0 / rxy : 1.0, s1 = rxy > 0.0 ? q1 / rxy : 0.0;
  double c = 1.0, s = 0.0;
  for (int mup = 0; mup <= mmax; ++mup) {
    phase[i * (mmax + 1) + mup] = make_float2(static_cast<float>(c), static_cast<float>(-s));
    const double t = c * c1 - s * s1;
    s = s * c1 + c * s1;
    c = t;
  }
}

// the angular grids with a compile-time kernel
template <typename F>
bool dispatch(int mmax, int mrso, F&& f) {
  if (mrso == 2 && mmax == 4)
    f(std::integral_constant<int, 4>{}, std::integral_constant<int, 2>{});
  else if (mrso == 2 && mmax == 5)
    f(std::integral_constant<int, 5>{}, std::integral_constant<int, 2>{});
  else
    return false;
  return true;
}

template <typename V>
V* upload(const std::vector<V>& h) {
  V* d = nullptr;
  MDFT_HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&d), std::max<size_t>(1, h.size()) * sizeof(V)));
  if (!h.empty()) MDFT_HIP_CHECK(hipMemcpy(d, h.data(), h.size() * sizeof(V), hipMemcpyHostToDevice));
  return d;
}

// where entry e of a half d table (rows (l, mu >= 0) of 2 mmax + 1 columns) and
// its mirror d_{-mu,-chi} = (-1)^{mu - chi} d_{mu,chi} go in the d blocks
template <int MMAX, int MRSO>
int place(int e) {
  using S = Sh<MMAX, MRSO>;
  const int h = e / S::W, c = e % S::W;
  int l = 0;
  while ((l + 1) * (l + 2) / 2 <= h) ++l;
  const int mu = h - l * (l + 1) / 2;
  if (l == 0 || c > 2 * l) return 0;
  const int to = S::dofs(l) + (l + mu) * S::CW + c, mirror = S::dofs(l) + (l - mu) * S::CW + 2 * l - c;
  return to | mirror << 12 | (((mu + c + l) & 1) ? kPlaceNeg : 0) | kPlaceValid;
}

}  // namespace

// A group of stars costs a CU the same however many of its stars exist, and a
// round of groups the chip: at mmax 5 12 us + 11.5 us a round of 8 stars per CU,
// where the star kernel takes 13 us + 6.9 ns a star.  So the last round decides
// (star kernel against this one, 2048 stars a round, FP32, us):
//   2197 stars 27.6 / 35.6, 2744 30.8 / 35.4, 3375 35.4 / 35.3, 3640 38.4 / 35.1,
//   4096 40.1 / 35.2, 4356 42.9 / 45.8, 4807 44.4 / 45.9, 4913 46.4 / 46.4,
//   5265 45.7 / 45.9, 6859 59.4 / 57.5, 9261 76.0 / 68.8, 15625 128 / 103
// and this kernel is taken where its rounds are filled to 0.82.  At mmax 4, whose
// stars are half as large and whose blocks share a CU, the sides meet at 17576
// stars (78.9 / 78.3; 15625 65.7 / 71.2, 19305 88.2 / 86.2, 21021 93.5 / 93.9,
// 24389 110 / 102, 35937 180 / 148).
bool OzGroup::serves(int mmax, int mrso, long nstars) {
  if (mrso != 2) return false;
  if (mmax == 4) return nstars >= 19000;
  if (mmax != 5) return false;
  int dev = 0, cus = 0;
  MDFT_HIP_CHECK(hipGetDevice(&dev));
  MDFT_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const long round = static_cast<long>(kStars) * std::max(1, cus), rounds = (nstars + round - 1) / round;
  return 100 * nstars >= 82 * rounds * round;
}

OzGroup::OzGroup(const ConvTables& tab, hipStream_t s)
    : nx_(tab.nx), ny_(tab.ny), nz_(tab.nz), mmax_(tab.mmax), mrso_(tab.mrso) {
  throw_if(!dispatch(mmax_, mrso_, [](auto, auto) {}), "OZ group pass: no kernel for this angular grid");
  const AngularGrid& g = tab.ang;
  const long nstars = static_cast<long>(nx_ / 2 + 1) * (ny_ / 2 + 1) * (nz_ / 2 + 1);
  int dev = 0;
  MDFT_HIP_CHECK(hipGetDevice(&dev));
  MDFT_HIP_CHECK(hipDeviceGetAttribute(&blocks_, hipDeviceAttributeMultiprocessorCount, dev));
  double* k = nullptr;
  try {
    dispatch(mmax_, mrso_, [&](auto mm, auto mr) {
      constexpr int MMAX = decltype(mm)::value, MRSO = decltype(mr)::value;
      using S = Sh<MMAX, MRSO>;
      throw_if(tab.np_new != S::terms(), "internal error: OZ term count");
      // c rows: terms by (chi, m, mu2, n, nu2) from (m, chi, mu2, n, nu2)
      std::vector<float2> c(static_cast<size_t>(tab.nq) * S::NCP, make_float2(0.f, 0.f));
      int at = 0;
      for (int chi = -MMAX; chi <= MMAX; ++chi)
        for (int m = std::abs(chi); m <= MMAX; ++m)
          for (int mu2 = 0; mu2 < S::km(m); ++mu2, at += S::ldc(chi))
            for (int q = 0; q < S::nins(chi); ++q) {
              const int ia = tab.ia_start[g.P(m, chi, mu2)] + q;
              for (int iq = 0; iq < tab.nq; ++iq) {
                const cd z = tab.ctab[static_cast<size_t>(ia) * tab.nq + iq];
                c[static_cast<size_t>(iq) * S::NCP + at + q] =
                    make_float2(static_cast<float>(z.real()), static_cast<float>(z.imag()));
              }
            }
      ctab_ = upload(c);
      std::vector<int> dc(S::NE);
      for (int e = 0; e < S::NE; ++e) dc[e] = place<MMAX, MRSO>(e);
      dcode_ = upload(dc);
      for (int cp = 0; cp < 2; ++cp) {
        std::vector<int> rec;
        for (int ip = 0; ip < g.np; ++ip) {
          const int m = g.m[ip], mup = g.mup[ip], mu2 = g.mu2[ip];
          if (cp && implied_projection(mup, g.mu[ip])) continue;
          int r = (S::rowbase(m, mu2) + mup + m) | (S::rowbase(m, mu2) - mup + m) << 10 | (mup + MMAX) << 20;
          if (mup & 1) r |= kRecOdd;
          if (cp && mu2 == 0 && mup > 0) r |= kRecFold;
          rec.push_back(r);
        }
        chrec_[cp] = upload(rec);
      }
    });
    std::vector<double> k3(tab.kx);
    k3.insert(k3.end(), tab.ky.begin(), tab.ky.end());
    k3.insert(k3.end(), tab.kz.begin(), tab.kz.end());
    k = upload(k3);
    MDFT_HIP_CHECK(hipMalloc(&meta_, nstars * sizeof(OzStarMeta)));
    MDFT_HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&phase_), nstars * (mmax_ + 1) * sizeof(float2)));
    hipLaunchKernelGGL(star_meta_kernel, dim3(static_cast<unsigned>((nstars + 255) / 256)), dim3(256), 0, s,
                       static_cast<OzStarMeta*>(meta_), phase_, k, nx_, ny_, ny_ / 2 + 1, nz_ / 2 + 1, nstars, mmax_,
                       tab.nq, tab.dq);
    MDFT_HIP_CHECK(hipGetLastError());
    MDFT_HIP_CHECK(hipStreamSynchronize(s));  // the k table is released below
    (void)hipFree(k);
  } catch (...) {
    if (k) (void)hipFree(k);
    release();
    throw;
  }
}

OzGroup::~OzGroup() {
  release();
}

void OzGroup::release() {
  for (void* q : {static_cast<void*>(ctab_), meta_, static_cast<void*>(phase_), static_cast<void*>(dcode_),
                  static_cast<void*>(chrec_[0]), static_cast<void*>(chrec_[1])})
    if (q) (void)hipFree(q);
}

void OzGroup::run(float2* p, const float* dtab, double chop_eps, int nbatch, bool compact, hipStream_t s,
                     hipEvent_t ev0, hipEvent_t ev1) const {
  dispatch(mmax_, mrso_, [&](auto mm, auto mr) {
    constexpr int MMAX = decltype(mm)::value, MRSO = decltype(mr)::value;
    using L = Lay<MMAX, MRSO>;
    {
      GroupArgs a;
      a.p = p;
      a.dtab = dtab;
      a.ctab = ctab_;
      a.meta = static_cast<const OzStarMeta*>(meta_);
      a.phase = phase_;
      a.dcode = dcode_;
      a.chrec = chrec_[compact ? 1 : 0];
      a.nx = nx_; a.ny = ny_; a.nz = nz_;
      a.hy = ny_ / 2 + 1;
      a.hz = nz_ / 2 + 1;
      a.nbatch = nbatch;
      a.nstars = (nx_ / 2 + 1) * a.hy * a.hz;
      a.ngroups = (a.nstars + kStars - 1) / kStars;
      a.chunk = (a.ngroups + kXcds - 1) / kXcds;
      a.N = static_cast<long>(nx_) * ny_ * nz_;
      a.pstride = a.N * nbatch;
      a.chop_eps = static_cast<float>(chop_eps);
      // persistent blocks: as many per XCD as its CUs hold, at most one per item
      const long slots = std::max<long>(1, std::min<long>(static_cast<long>(a.chunk) * nbatch, static_cast<long>(blocks_) / kXcds * L::per_cu));
      const unsigned nb = static_cast<unsigned>(slots * kXcds);
      auto go = [&](auto kernel) {
        if (ev0 || ev1)
          hipExtLaunchKernelGGL(kernel, dim3(nb), dim3(kThreads), static_cast<std::uint32_t>(L::total), s, ev0, ev1, 0u, a);
        else
          hipLaunchKernelGGL(kernel, dim3(nb), dim3(kThreads), L::total, s, a);
        MDFT_HIP_CHECK(hipGetLastError());
      };
      if (compact)
        go(oz_group_kernel<MMAX, MRSO, true>);
      else
        go(oz_group_kernel<MMAX, MRSO, false>);
    }
  });
}

}  // namespace mdft
