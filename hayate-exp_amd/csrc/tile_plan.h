// The plan of a prompt-row product (tiles.hip): which tile, and into how many
// pieces of k it is split. Host code only.
#pragma once

#include <math.h>

#include <cstdint>

namespace hy {

constexpr int kStepK = 64;
// Row tiles that share a pass over the weights, at most. An XCD's workgroups are
// neighbours in this order, so its L2 serves their common rows.
constexpr int kRowGroup = 10;

// Each tile's time per step of 64 k with the chip full, measured on MI355X. The
// large ones do more per byte that crosses LDS, the small ones leave fewer CUs
// idle when there are few rows; a split fills the chip where the outputs alone
// do not (the down projection of 512 rows: 40 tiles of 256 x 128, 41 us in 5
// pieces, 123 whole). The plan is the least of
//   rounds * steps * step time (or the weights' bytes at 4.2 TB/s, slower by the
//   root of the idle part when CUs are idle) + 2.5 us + 0.4 us per MB of partials,
//   if split.
// Measured at 64, 128, 300, 512, 1024 and 2064 rows of the three products of a
// 2560-wide block over 12 tiles x 10 splits, it picks one within 10 % of the best.
struct TileShape {
  int bm, bn;
  float step_us;
};
constexpr TileShape kShapes[] = {{64, 128, 0.42f},  {128, 96, 0.50f},  {128, 128, 0.58f},
                                 {128, 192, 0.85f}, {256, 128, 0.97f}, {256, 160, 1.14f}};
constexpr int kNumShapes = sizeof(kShapes) / sizeof(kShapes[0]);
constexpr int kCus = 256, kMaxSplits = 16, kMinSteps = 4;

struct TilePlan {
  int shape, row_tiles, col_tiles, splits, row_group;
  int64_t bytes;  // partials
};

inline TilePlan plan_tiles(int m, int n, int k, bool gated) {
  TilePlan best{};
  float best_us = -1.0f;
  const int steps = k / kStepK;
  const float weights_us = (gated ? 2.0f : 1.0f) * 2.0f * n * k / 4.2e6f;
  for (int s = 0; s < kNumShapes; ++s) {
    const int cols = gated ? kShapes[s].bn / 2 : kShapes[s].bn;
    const int row_tiles = (m + kShapes[s].bm - 1) / kShapes[s].bm;
    const int col_tiles = (n + cols - 1) / cols;
    const int64_t tiles = static_cast<int64_t>(row_tiles) * col_tiles;
    for (int splits = 1; splits <= kMaxSplits; ++splits) {
      // a split is for chips that the outputs do not fill
      if (splits > 1 && (tiles * splits > kCus || steps / splits < kMinSteps)) break;
      const int64_t rounds = (tiles * splits + kCus - 1) / kCus;
      const int64_t bytes = splits > 1 ? tiles * splits * kShapes[s].bm * kShapes[s].bn * 4 : 0;
      float us = static_cast<float>(rounds) * ((steps + splits - 1) / splits) * kShapes[s].step_us;
      const float busy = static_cast<float>(tiles * splits < kCus ? tiles * splits : kCus) / kCus;
      const float read_us = weights_us / sqrtf(busy);
      if (us < read_us) us = read_us;
      if (splits > 1) us += 2.5f + 0.4e-6f * static_cast<float>(bytes);
      if (best_us < 0.0f || us < best_us) {
        best_us = us;
        // equal groups: a short last one would read all weights for little
        const int groups = (row_tiles + kRowGroup - 1) / kRowGroup;
        best = {s, row_tiles, col_tiles, splits, (row_tiles + groups - 1) / groups, bytes};
      }
    }
  }
  return best;
}

}  // namespace hy
