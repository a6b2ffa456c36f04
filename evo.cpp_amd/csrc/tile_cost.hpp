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
// `load` is what a step slows down by as the whole chip fills.
struct TileCost {
  float launch, epilogue, load;
  int slots;
  float step[3];
};

// `weight_bytes` come from HBM at the measured copy rate, 5 TB/s.
inline double tile_us(const TileCost &c, double blocks, double steps, double weight_bytes) {
  const double per_round = 256.0 * c.slots;
  const double rounds = std::floor(blocks / per_round);
  const int rest = static_cast<int>(std::ceil((blocks - rounds * per_round) / 256.0));
  double us = c.launch + rounds * (c.epilogue + steps * c.step[c.slots - 1]) +
              c.load * steps * blocks / 256.0;
  if (rest > 0)
    us += c.epilogue + steps * c.step[rest - 1];
  return std::max(us, 3.0 + weight_bytes / 5.0e6);
}

}  // namespace evo::hip
