// The OZ pass over groups of consecutive stars on the matrix cores (see
// mdft_oz_group.hip).
#pragma once

#include <memory>

#include "mdft_device.hpp"

namespace mdft {

// The per-star tables and the launch of the FP32 pass.  A
// star is the set of q = (+-kx, +-ky, +-kz); star (|ix|, |iy|, |iz|) has the
// index (|ix| (ny/2 + 1) + |iy|) (nz/2 + 1) + |iz|, the order of oz_stars.
class OzGroup {
 public:
  // whether this pass is the faster one for the grid
  static bool serves(int mmax, int mrso, long nstars);
  OzGroup(const ConvTables& tab, hipStream_t s);
  ~OzGroup();
  OzGroup(const OzGroup&) = delete;
  OzGroup& operator=(const OzGroup&) = delete;
  // dtab: one half d table per star (rows of 2 mmax + 1); p, nbatch, compact
  // and the events as ConvDevice::oz_pass
  void run(float2* p, const float* dtab, double chop_eps, int nbatch, bool compact, hipStream_t s, hipEvent_t ev0,
           hipEvent_t ev1) const;

 private:
  void release();
  int nx_, ny_, nz_, mmax_, mrso_;
  int blocks_ = 0;            // CUs of the device
  float2* ctab_ = nullptr;   // c(q) rows, chi-major terms
  void* meta_ = nullptr;      // per star: c(q) row, lerp weights
  float2* phase_ = nullptr;  // per star: e^{-i mup phi} of (|kx|, |ky|), mup = 0 .. mmax
  int* dcode_ = nullptr;      // LDS places of the half d table's entries
  int* chrec_[2] = {nullptr, nullptr};  // per channel (full, compact): its LDS row and (m, mup, mu2)
};

}  // namespace mdft
