// SPDX-License-Identifier: Apache-2.0
// C entry points for this repository's tests, in a library of their own
// (lib/libevo_hip_testing.so): the launch rules as functions of the sizes, and
// products on a given block tile. No part of the product's interface.
#include <hip/hip_runtime.h>

#include <chrono>

#include "gemm_tile.hpp"
#include "launch_rules.hpp"
#include "ops.hpp"

#define EVO_TEST_API extern "C" __attribute__((visibility("default")))

EVO_TEST_API unsigned evo_test_hcs_stream_segment(size_t width, size_t length, int f32_rows,
                                                  int exact, int f32_out) {
  return evo::hip::hcs_stream_segment(width, length, f32_rows != 0, exact != 0, f32_out != 0);
}

EVO_TEST_API int evo_test_hcm_stream_two_groups(size_t group_size, size_t length, int taps,
                                                int f32, int caches) {
  return evo::hip::hcm_stream_two_groups(group_size, length, taps, f32 != 0, caches != 0) ? 1 : 0;
}

// Tile of a dense product (-1: 256 x 256); its K parts and tail tiles.
EVO_TEST_API int evo_test_linear_plan(size_t m, size_t n, size_t k, int split, int gated,
                                      size_t workspace_bytes, int *parts, size_t *tail) {
  const auto plan =
      evo::hip::plan_linear(m, n, k, split != 0, gated != 0, workspace_bytes, false);
  *parts = plan.choice.splits;
  *tail = plan.tail;
  return plan.choice.tile;
}
// Mean host time of that choice, in ns.
EVO_TEST_API double evo_test_linear_plan_ns(size_t m, size_t n, size_t k, size_t workspace_bytes,
                                            int calls) {
  using Clock = std::chrono::steady_clock;
  volatile int tile = 0;
  const auto start = Clock::now();
  for (int i = 0; i < calls; ++i)
    tile = evo::hip::plan_linear(m, n, k, true, false, workspace_bytes, false).choice.tile;
  return std::chrono::duration<double, std::nano>(Clock::now() - start).count() / calls;
}
EVO_TEST_API int evo_test_linear_tiles(void) { return evo::hip::kGemmTiles; }
EVO_TEST_API int evo_test_fp8_tiles(void) { return evo::hip::kFp8TileCount; }
EVO_TEST_API int evo_test_fp8_tile(size_t m, size_t n, size_t k, int mode) {
  return evo::hip::choose_fp8_tile(m, n, k, mode == evo::hip::kFp8MfmaK32);
}

// out = x . w^T (+ residual) on block tile `tile` with K in `parts` parts
// (workspace: parts x m x n floats when parts > 1); f16: x_hi and w are FP16.
// k % (32 * parts) == 0 and k / parts no less than the tile's step, which is
// at most 128. Returns 0 on success.
EVO_TEST_API int evo_test_linear_on_tile(int tile, int parts, const uint16_t *x_hi,
                                         const uint16_t *x_lo, int f16, const uint16_t *w,
                                         const float *residual, size_t m, size_t n, size_t k,
                                         float *out, float *workspace, void *stream) {
  using namespace evo::hip;
  if (m == 0 || n == 0 || parts < 1 || k % (32 * static_cast<size_t>(parts)) != 0 ||
      k / parts < 128 || (parts > 1 && (workspace == nullptr || n % 4 != 0)) ||
      (f16 != 0 && x_lo != nullptr))
    return 1;
  const auto s = static_cast<hipStream_t>(stream);
  const Epilogue whole{residual != nullptr ? kGemmResidual : kGemmStore, nullptr, residual, 0, 0};
  const Epilogue part{kGemmStore, nullptr, nullptr, 0, 0};
  const int width = static_cast<int>(n);
  const TileCall call{x_hi, x_lo, static_cast<int>(k), f16 != 0, w, static_cast<int>(m), width,
                      static_cast<int>(k), parts, parts > 1 ? workspace : out,
                      parts > 1 ? m * n : 0, nullptr, nullptr, width, parts > 1 ? part : whole};
  if (!gemm_tile(tile, call, s).ok())
    return 1;
  if (parts == 1)
    return 0;
  return split_k_finish(SplitPartials{workspace, parts, m * n, nullptr, residual}, out, m, n, s)
                 .ok() ? 0 : 1;
}

// The gated product (w12 from evo_hip_pack_mlp, n rows) on a block tile: split
// planes [m, inner], out_lo may be null.
EVO_TEST_API int evo_test_gated_on_tile(int tile, const uint16_t *x_hi, const uint16_t *x_lo,
                                        const uint16_t *w12, size_t m, size_t width, size_t inner,
                                        int gelu, uint16_t *out_hi, uint16_t *out_lo,
                                        void *stream) {
  using namespace evo::hip;
  const size_t n = (inner + 31) / 32 * 64;
  // (Tile 0 is 16 columns wide: it holds no l1 and l2 pair.)
  if (tile == 0 || m == 0 || inner == 0 || width % 32 != 0 || width < 128)
    return 1;
  const Epilogue epi{kGemmGated, nullptr, nullptr, gelu, static_cast<int>(inner)};
  const TileCall call{x_hi, x_lo, static_cast<int>(width), false, w12, static_cast<int>(m),
                      static_cast<int>(n), static_cast<int>(width), 1, nullptr, 0, out_hi, out_lo,
                      static_cast<int>(inner), epi};
  return gemm_tile(tile, call, static_cast<hipStream_t>(stream)).ok() ? 0 : 1;
}

// evo_hip_fp8_linear_bf16's MFMA product (mode 0 or 1) on a block tile.
EVO_TEST_API int evo_test_fp8_on_tile(int tile, const uint8_t *x, const uint8_t *w, uint16_t *out,
                                      size_t m, size_t n, size_t k, float scale, int mode,
                                      void *stream) {
  if (m == 0 || n == 0 || k == 0 || k % 128 != 0 || (mode != 0 && mode != 1))
    return 1;
  return evo::hip::fp8_linear_on_tile(tile, x, w, out, m, n, k, scale,
                                      static_cast<evo::hip::Fp8Mode>(mode),
                                      static_cast<hipStream_t>(stream)).ok() ? 0 : 1;
}
