// SPDX-License-Identifier: Apache-2.0
// Small-tile dense linears (gemm_tile.hip), the part of gemm_bf16w below the
// 256 x 256 tiles.
#pragma once

#include <hip/hip_runtime.h>

#include "gemm_epilogue.hpp"

namespace evo::hip {

// A block tile of gemm_tile.hip (-1: the 256 x 256 tile is the cheaper one)
// and the number of K parts it runs as.
struct TileChoice {
  int tile = -1;
  int splits = 1;
};
// The cheapest tile for C[M,N] of K by measured cost. `large_parts`: the K
// parts the 256 x 256 tile would run as; workspace_bytes (0: none) bounds the
// F32 partials of a split; `deferred`: the consumer sums the partials.
TileChoice choose_gemm_tile(size_t M, size_t N, size_t K, bool split, bool gated,
                            size_t large_parts, size_t workspace_bytes, bool deferred);

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
