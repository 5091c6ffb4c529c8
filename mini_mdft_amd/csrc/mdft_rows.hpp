// Row arithmetic of the proj2angl epilogue (mdft_p2a_wave.hip), host code too.
#pragma once

namespace mdft {

// A block of THREADS threads walks ROWS consecutive rows of NJK values: thread
// (sub, col) = (tid / NJK, tid mod NJK), sub < kG, takes column col of the rows
// sub, sub + kG, ...  The last block of a field ends at row last < ROWS: steps
// past it, and threads whose first row is past it, stay on a row that exists.
template <int NJK, int THREADS, int ROWS>
struct RowWalk {
  static constexpr int kG = THREADS / NJK < 16 ? THREADS / NJK : 16;  // rows of one step of the block
  static constexpr int kSteps = (ROWS + kG - 1) / kG;
  static constexpr int first(int sub, int last) { return sub < last ? sub : last; }
  // steps of kG rows from the first one to the thread's last
  static constexpr int reach(int sub, int last) { return (last - first(sub, last)) / kG; }
  static constexpr int row(int sub, int u, int last) {
    const int n = reach(sub, last);
    return first(sub, last) + (u < n ? u : n) * kG;
  }
};

}  // namespace mdft
