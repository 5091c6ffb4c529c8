// Host check of RowWalk (mdft_rows.hpp): on every angular grid of the kernel and
// for every last row of a block, each thread's every step reads a row that
// exists, and the rows stored (sub <= last, steps up to reach) are 0 .. last,
// each once.
#include <cstdio>
#include <vector>

#include "mdft_rows.hpp"

static int bad = 0;

template <int MMAX, int MRSO>
void check() {
  constexpr int kRows = 64, kNmu2 = MMAX / MRSO + 1, kNjk = (2 * MMAX + 1) * (2 * (MMAX / MRSO) + 1);
  using Walk = mdft::RowWalk<kNjk, 64 * kNmu2, kRows>;
  for (int last = 0; last < kRows; ++last) {
    std::vector<int> seen(kRows, 0);
    for (int sub = 0; sub < Walk::kG; ++sub)
      for (int u = 0; u < Walk::kSteps; ++u) {
        const int row = Walk::row(sub, u, last);
        if (row < 0 || row > last) {
          if (++bad <= 5)
            std::printf("mmax %d mrso %d: last row %d, thread row %d, step %d reads row %d\n", MMAX, MRSO, last, sub, u,
                        row);
          continue;
        }
        if (sub <= last && u <= Walk::reach(sub, last)) ++seen[row];
      }
    for (int r = 0; r <= last; ++r)
      if (seen[r] != 1) {
        if (++bad <= 5) std::printf("mmax %d mrso %d: last row %d, row %d stored %d times\n", MMAX, MRSO, last, r, seen[r]);
      }
  }
}

int main() {
  check<1, 1>();
  check<2, 1>();
  check<3, 1>();
  check<1, 2>();
  check<2, 2>();
  check<3, 2>();
  check<4, 2>();
  check<5, 2>();
  check<6, 2>();
  std::printf("%d failed\n", bad);
  return bad ? 1 : 0;
}
