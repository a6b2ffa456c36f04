// SPDX-License-Identifier: Apache-2.0
// Small-tile dense linears (gemm_tile.hip), the part of gemm_bf16w below the
// 256 x 256 tiles.
#pragma once

#include <hip/hip_runtime.h>

#include "gemm_epilogue.hpp"
#include "launch_rules.hpp"

namespace evo::hip {

struct TileCall {
  const uint16_t *a_hi, *a_lo;  // a_lo null: one plane
  int lda;
  bool f16;           // FP16 activation and weight
  const uint16_t *W;  // row stride K
  int M, N, K;
  int splits;  // K parts of K / splits each, part s stored at C + s * c_split
  float *C;
  size_t c_split;
  uint16_t *c_hi, *c_lo;  // gated output planes
  int ldc;
  Epilogue epi;
};
// K % 32 == 0, K / splits a multiple of 32 and no less than the tile's step
// (choose_gemm_tile's conditions).
Status gemm_tile(int tile, const TileCall &call, hipStream_t stream);

}  // namespace evo::hip
