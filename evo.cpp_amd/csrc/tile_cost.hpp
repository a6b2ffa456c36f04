// SPDX-License-Identifier: Apache-2.0
// Measured cost of a tiled product, by which the dense linears choose their
// block tile (host code).
#pragma once

#include <algorithm>
#include <cmath>

namespace evo::hip {

// Time of a launch on one tile, in us: launch + rounds * (epilogue + steps *
// step) + load * steps * blocks / 256, where a round fills each of the 256
// CUs with `slots` blocks (step[r - 1]: a K step of a CU's r blocks) and
// `load` is what a step slows down by as the whole chip fills; 1 us + the
// weight's bytes at `rate` TB/s, what the tile streams from HBM; and the bytes
// that the XCDs' L2s read at `fill` TB/s (0: not its bound). All fitted on
// weights that no cache holds.
struct TileCost {
  float launch, epilogue, load;
  int slots;
  float step[3];
  float rate = 5.4F, fill = 0.0F;
};

// The bounds join in a 6-norm: under a hard maximum every tile that stays
// below the bytes' time cost the same, and the order of the table picked among
// them (17 to 32 rows of 22528 x 4096: 44 to 49 us against 39).
inline double tile_us(const TileCost &c, double blocks, double steps, double weight_bytes,
                      double fill_bytes = 0.0) {
  const double per_round = 256.0 * c.slots;
  const double rounds = std::floor(blocks / per_round);
  const int rest = static_cast<int>(std::ceil((blocks - rounds * per_round) / 256.0));
  double us = c.launch + rounds * (c.epilogue + steps * c.step[c.slots - 1]) +
              c.load * steps * blocks / 256.0;
  if (rest > 0)
    us += c.epilogue + steps * c.step[rest - 1];
  const double bytes_us = 1.0 + weight_bytes / (1.0e6 * c.rate);
  const double fill_us = c.fill > 0.0F ? fill_bytes / (1.0e6 * c.fill) : 0.0;
  const double longest = std::max({us, bytes_us, fill_us});
  double sum = 0.0;
  for (const double bound : {us, bytes_us, fill_us}) {
    const double ratio = bound / longest, cube = ratio * ratio * ratio;
    sum += cube * cube;
  }
  return longest * std::cbrt(std::sqrt(sum));
}

}  // namespace evo::hip
