// Test helper: for tiles of argv[1] indices a run over operands of T .. argv[2]
// indices, one line per tile, "count i0" and then "index,owned" for every
// element of every lane row's run, as novaq_split_index.h has them.  Built with
// g++ by tests/test_split_index.py.
#include <cstdio>
#include <cstdlib>

#include "../../novann_amd/csrc/novaq_split_index.h"

int main(int argc, char** argv) {
  using namespace novaq::split_detail;
  const int T = argc > 1 ? std::atoi(argv[1]) : 2, most = argc > 2 ? std::atoi(argv[2]) : 200;
  for (int count = T; count <= most; ++count)
    for (int i0 = 0; i0 < count; i0 += 16 * T) {
      const int last = col_last(T, count, i0);
      std::printf("%d %d", count, i0);
      for (int r = 0; r < 16; ++r)
        for (int t = 0; t < T; ++t)
          std::printf(" %d,%d", col_index(T, last, t, r), (int)col_owns(T, last, t, r));
      std::printf("\n");
    }
  return 0;
}
