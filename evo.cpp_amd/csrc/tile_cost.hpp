// SPDX-License-Identifier: Apache-2.0
// Measured cost of a tiled product, by which the dense linears choose their
// block tile (host code).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

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
// them (17 to 32 rows of 22528 x 4096: 44 to 49 us against 39). A candidate
// that can't come out below `limit` returns any time of at least `limit`: each
// call weighs up to 40 of them, and its launch waits for that.
inline float tile_us(const TileCost &c, uint32_t blocks, uint32_t steps, float weight_bytes,
                     float fill_bytes, float limit) {
  const uint32_t per_round = 256U * static_cast<uint32_t>(c.slots);
  const uint32_t rounds = blocks / per_round, rest = (blocks - rounds * per_round + 255U) / 256U;
  const float k_steps = static_cast<float>(steps);
  float us = c.launch + static_cast<float>(rounds) * (c.epilogue + k_steps * c.step[c.slots - 1]) +
             c.load * k_steps * static_cast<float>(blocks) * (1.0F / 256.0F);
  if (rest > 0)
    us += c.epilogue + k_steps * c.step[rest - 1];
  const float bytes_us = 1.0F + weight_bytes / (1.0e6F * c.rate);
  const float fill_us = c.fill > 0.0F ? fill_bytes / (1.0e6F * c.fill) : 0.0F;
  const float longest = std::max({us, bytes_us, fill_us});
  if (longest >= limit)
    return longest;
  float sum = 0.0F;
  for (const float bound : {us, bytes_us, fill_us}) {
    const float ratio = bound / longest, cube = ratio * ratio * ratio;
    sum += cube * cube;
  }
  return longest * std::cbrt(std::sqrt(sum));
}

}  // namespace evo::hip
