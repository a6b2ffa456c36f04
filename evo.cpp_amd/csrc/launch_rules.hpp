// SPDX-License-Identifier: Apache-2.0
// The rules by which launches choose their shape, as functions of the sizes
// (host code; the reasons and measurements stand at the definitions). The
// dispatches call them, and so do the tests, through testing.cpp.
#pragma once

#include <cstddef>

namespace evo::hip {

// A block tile of gemm_tile.hip (-1: the 256 x 256 tile of gemm.hip) and the
// number of K parts it runs as.
struct TileChoice {
  int tile = -1;
  int splits = 1;
};
// The cheapest tile for C[M,N] of K by measured cost. `large_parts`: the K
// parts the 256 x 256 tile would run as; workspace_bytes (0: none) bounds the
// F32 partials of a split; `deferred`: the consumer sums the partials.
TileChoice choose_gemm_tile(size_t M, size_t N, size_t K, bool split, bool gated,
                            size_t large_parts, size_t workspace_bytes, bool deferred);
constexpr int kGemmTiles = 10;

// How gemm_bf16w runs a product of more than four rows and K % 32 == 0:
// `split`: hi + lo activation planes; workspace_bytes: of a 16-byte aligned
// workspace, 0 without one; `deferred` as above. tail: trailing 256 x 256
// tiles that run as two K halves (choice.tile == -1).
struct LinearPlan {
  TileChoice choice;
  size_t tail = 0;
};
LinearPlan plan_linear(size_t M, size_t N, size_t K, bool split, bool gated,
                       size_t workspace_bytes, bool deferred);

// Block tile of an MFMA-mode FP8 product of more than four rows (fp8.hip).
int choose_fp8_tile(size_t M, size_t N, size_t K, bool k32);
constexpr int kFp8TileCount = 6;

// Rows per segment of the HCS row stream (hyena.hip); exact: a short FIR of 3
// and 7 taps.
unsigned hcs_stream_segment(size_t width, size_t length, bool f32_rows, bool exact, bool f32_out);

// Whether the HCM row stream takes filter groups that are no multiple of 16
// (hyena.hip), rows and outputs aligned.
bool hcm_stream_two_groups(size_t group_size, size_t length, int taps, bool f32, bool caches);

}  // namespace evo::hip
