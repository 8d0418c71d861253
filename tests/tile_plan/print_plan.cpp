// Plans of the prompt-row products named on stdin, lines "m n k gated": prints
// shape, its rows and columns of outputs, and the splits. With an argument: every
// (shape, gated, split) that any product of a wide range gets.
#include <cstdio>
#include <set>
#include <tuple>

#include "../../hayate-exp_amd/csrc/tile_plan.h"

int main(int argc, char **) {
  if (argc > 1) {
    std::set<std::tuple<int, int, int>> seen;
    for (int m = 1; m <= 16384; m += m < 200 ? 1 : m / 37)
      for (int k = 64; k <= 30000; k += k < 1024 ? 64 : k / 8 / 64 * 64)
        for (int n = 4; n <= 32768; n += n < 128 ? 12 : n / 9 / 4 * 4)
          for (int gated = 0; gated < 2; ++gated) {
            const auto p = hy::plan_tiles(m, n, k, gated);
            seen.insert({p.shape, gated, p.splits > 1});
          }
    for (const auto &[shape, gated, split] : seen) std::printf("%d %d %d\n", shape, gated, split);
    return 0;
  }
  int m, n, k, gated;
  while (std::scanf("%d %d %d %d", &m, &n, &k, &gated) == 4) {
    const auto p = hy::plan_tiles(m, n, k, gated);
    const auto &s = hy::kShapes[p.shape];
    std::printf("%d %d %d %d\n", p.shape, s.bm, gated ? s.bn / 2 : s.bn, p.splits);
  }
}
