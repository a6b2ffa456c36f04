// SPDX-License-Identifier: Apache-2.0
// Dense linears on small block tiles: the products C[M,N] = A[M,K] . W[N,K]^T
// of 5 to a few thousand rows, where 256 x 256 tiles (gemm.hip) leave most
// CUs idle or multiply padding. Same operands, split-plane products and
// epilogues as gemm.hip.
//
// Few rows are bound by the weight's bytes, so every CU has to stream its own
// weight rows: a block tile is as narrow as the shape needs to fill 256 CUs
// without splitting K across blocks (no workspace). Operands reach LDS by DMA
// in row pieces of 128 or 256 bytes (64-byte pieces, what a 32-K step reads,
// move 24-45 bytes per clock and CU from L2, 128-byte ones 58-60), 3-6 steps
// deep, so the LDS holds up to 150 KB of reads in flight per CU. (Fragments
// loaded straight to registers, 16 rows x 64 bytes per instruction, reached
// 16-20 bytes per clock: 62 us against 37 for 61 rows of 4096 x 11264.)
// The 32-K slices of a step go to different waves, which halves or quarters
// the fragment reads a wave shape of the whole step would repeat; their sums
// meet in LDS at the end.
//
// Measured (MI355X, split planes, weights that no cache holds; floor: their
// bytes at 5.4 TB/s), against 256 x 256 tiles without a workspace:
//   N = 22528, K = 4096: 5 rows 154 -> 38 us, 61 rows 154 -> 50, 200 rows
//     166 -> 89, 700 rows 351 -> 255 (floor 34)
//   N = 4096, K = 11264: 5 rows 392 -> 22 us, 61 rows 393 -> 38, 300 rows
//     416 -> 97, 1000 rows 434 -> 155 (floor 17)
//   N = K = 1920: 61 rows 80 -> 8 us, 1000 rows 90 -> 23.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "gemm_epilogue.hpp"
#include "gemm_tile.hpp"
#include "tile_cost.hpp"

namespace evo::hip {
namespace {

// One block tile. kSeg K elements (64 or 128: 128- or 256-byte row pieces)
// are staged per step; the waves are kWK (32-K slices of a step) x kWM x kWN.
template <int kBM_, int kBN_, int kSeg_, int kWK_, int kWM_, int kWN_, int kStages_>
struct TileShape {
  static constexpr int kBM = kBM_, kBN = kBN_, kSeg = kSeg_, kWK = kWK_, kWM = kWM_, kWN = kWN_,
                       kStages = kStages_;
  static constexpr int kWaves = kWK * kWM * kWN;
  static constexpr int kMI = kBM / 16 / kWM, kNJ = kBN / 16 / kWN;
};

// LDS of one row of kUnits 16-byte units: 16 consecutive rows read at one
// logical unit (a fragment's rows) fall on 16 distinct 16-byte bank groups.
template <int kUnits> __device__ inline int tile_unit(int row, int unit) {
  return row * kUnits + (unit ^ (kUnits == 8 ? ((row >> 1) & 7) : (row & 15)));
}

template <typename T, bool kSplit, bool kF16>
__global__ __launch_bounds__(T::kWaves * 64) void gemm_tile_kernel(
    const uint16_t *__restrict__ a_hi, const uint16_t *__restrict__ a_lo, int lda,
    const uint16_t *__restrict__ W, int ldw, int M, int N, int K, float *__restrict__ C,
    size_t c_split, uint16_t *__restrict__ c_hi, uint16_t *__restrict__ c_lo, int ldc,
    const Epilogue epi) {
  using Frag = std::conditional_t<kF16, f16x8, bf16x8>;
  constexpr int kPlanes = kSplit ? 2 : 1;
  constexpr int kBM = T::kBM, kBN = T::kBN, kUnits = T::kSeg / 8;
  constexpr int kMI = T::kMI, kNJ = T::kNJ, kTM = kBM / 16, kTN = kBN / 16;
  constexpr int kStageBytes = (kPlanes * kBM + kBN) * T::kSeg * 2;
  constexpr int kDma = kStageBytes / 1024 / T::kWaves;  // per wave and step
  static_assert(kStageBytes % (1024 * T::kWaves) == 0 && kDma * (T::kStages - 2) < 64, "DMA split");
  extern __shared__ __attribute__((aligned(16))) uint8_t tile_lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave_k = wave % T::kWK, wave_mn = wave / T::kWK;
  const int wave_m = wave_mn / T::kWN, wave_n = wave_mn % T::kWN;
  const int r16 = lane & 15, g = lane >> 4;
  const bool gated = epi.mode == kGemmGated;
  const int m_blocks = (M + kBM - 1) / kBM;
  const int linear = xcd_linear(blockIdx.x, gridDim.x);
  const int m0 = (linear % m_blocks) * kBM, block_n = linear / m_blocks;
  {
    const size_t k_first = static_cast<size_t>(blockIdx.y) * K;
    a_hi += k_first;
    if (kSplit)
      a_lo += k_first;
    W += k_first;
    C += blockIdx.y * c_split;
  }
  // Weight row of tile column x. Gated: the first half of the tile holds the
  // l1 rows, the second half the l2 rows of the same kBN / 2 gated columns.
  auto weight_row = [&](int x) {
    if (!gated)
      return block_n * kBN + x;
    const int half = x < kBN / 2 ? 0 : 1;
    const int column = block_n * (kBN / 2) + x - half * (kBN / 2);
    return (column / 32) * 64 + half * 32 + column % 32;
  };
  // This lane's DMA sources: rows of A hi, (A lo,) W in stage order.
  const uint16_t *src[kDma];
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int flat = (wave * kDma + i) * 64 + lane;
    const int row = flat / kUnits;
    const int unit = tile_unit<kUnits>(row, flat % kUnits) - row * kUnits;
    const uint16_t *base;
    if (row < kBM)
      base = a_hi + static_cast<size_t>(min(m0 + row, M - 1)) * lda;
    else if (kSplit && row < 2 * kBM)
      base = a_lo + static_cast<size_t>(min(m0 + row - kBM, M - 1)) * lda;
    else
      base = W + static_cast<size_t>(min(weight_row(row - kPlanes * kBM), N - 1)) * ldw;
    src[i] = base + unit * 8;
  }
  const int steps = (K + T::kSeg - 1) / T::kSeg;
  // The last step of a K that is no multiple of kSeg reads the last kSeg
  // elements and skips the 32-K slices the step before has multiplied.
  auto issue = [&](int step) {
    uint8_t *stage = tile_lds + (step % T::kStages) * kStageBytes;
    const int k0 = min(step * T::kSeg, K - T::kSeg);
#pragma unroll
    for (int i = 0; i < kDma; ++i)
      dma16(src[i] + k0, stage + (wave * kDma + i) * 1024);
  };

  f32x4 acc[kMI][kNJ];
#pragma unroll
  for (int i = 0; i < kMI; ++i)
#pragma unroll
    for (int j = 0; j < kNJ; ++j)
      acc[i][j] = f32x4{0.0F, 0.0F, 0.0F, 0.0F};
#pragma unroll
  for (int s = 0; s + 1 < T::kStages; ++s)
    if (s < steps)
      issue(s);
  for (int s = 0; s < steps; ++s) {
    wait_steps<kDma, T::kStages - 2>(steps - 1 - s);
    // Every wave's DMA of step s has landed, and every wave has left the
    // buffer of step s - 1, which the next issue overwrites.
    __syncthreads();
    if (s + T::kStages - 1 < steps)
      issue(s + T::kStages - 1);
    const uint8_t *stage = tile_lds + (s % T::kStages) * kStageBytes;
    const int skip = s + 1 < steps ? 0 : (steps * T::kSeg - K) / 32;
#pragma unroll
    for (int h = 0; h < T::kSeg / 32 / T::kWK; ++h) {
      const int slice = h * T::kWK + wave_k;
      if (slice < skip)
        continue;
      auto fragment = [&](int row) {
        return *reinterpret_cast<const Frag *>(stage + tile_unit<kUnits>(row, slice * 4 + g) * 16);
      };
      Frag b[kNJ], ah[kMI], al[kMI];
#pragma unroll
      for (int j = 0; j < kNJ; ++j)
        b[j] = fragment(kPlanes * kBM + (wave_n * kNJ + j) * 16 + r16);
#pragma unroll
      for (int i = 0; i < kMI; ++i) {
        ah[i] = fragment((wave_m * kMI + i) * 16 + r16);
        if (kSplit)
          al[i] = fragment(kBM + (wave_m * kMI + i) * 16 + r16);
      }
#pragma unroll
      for (int i = 0; i < kMI; ++i)
#pragma unroll
        for (int j = 0; j < kNJ; ++j) {
          if constexpr (kF16)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], b[j], acc[i][j], 0, 0, 0);
          else
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], b[j], acc[i][j], 0, 0, 0);
        }
      if constexpr (kSplit) {
#pragma unroll
        for (int i = 0; i < kMI; ++i)
#pragma unroll
          for (int j = 0; j < kNJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], b[j], acc[i][j], 0, 0, 0);
      }
    }
  }

  // The block's 16 x 16 tiles through LDS, [wave_k][tile row][tile column]:
  // the K slices are summed in order, and a gated pair meets in one lane.
  __syncthreads();
  f32x4 *part = reinterpret_cast<f32x4 *>(tile_lds);
#pragma unroll
  for (int i = 0; i < kMI; ++i)
#pragma unroll
    for (int j = 0; j < kNJ; ++j)
      part[((wave_k * kTM + wave_m * kMI + i) * kTN + wave_n * kNJ + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  auto total = [&](int ti, int tj) {
    f32x4 v = part[(ti * kTN + tj) * 64 + lane];
#pragma unroll
    for (int w = 1; w < T::kWK; ++w) {
      const f32x4 p = part[((w * kTM + ti) * kTN + tj) * 64 + lane];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = v[e] + p[e];
    }
    return v;
  };
  // Accumulator e of a tile: row 4 * (lane / 16) + e, column lane % 16.
  if constexpr (kTN % 2 == 0) {
    if (gated) {
      for (int t = wave; t < kTM * (kTN / 2); t += T::kWaves) {
        const int ti = t / (kTN / 2), tj = t % (kTN / 2);
        const f32x4 first = total(ti, tj), second = total(ti, tj + kTN / 2);
        const int col = block_n * (kBN / 2) + tj * 16 + r16;
        if (col >= epi.gated_width)
          continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = m0 + ti * 16 + 4 * g + e;
          if (row < M) {
            const float value = (epi.gelu ? gelu_erf(first[e]) : first[e]) * second[e];
            const size_t index = static_cast<size_t>(row) * ldc + col;
            const uint16_t hi = f32_to_bf16(value);
            c_hi[index] = hi;
            if (c_lo != nullptr)
              c_lo[index] = f32_to_bf16(value - bf16_to_f32(hi));
          }
        }
      }
      return;
    }
  }
  const bool bias_mode = epi.mode == kGemmBias || epi.mode == kGemmBiasResidual;
  const bool res_mode = epi.mode == kGemmResidual || epi.mode == kGemmBiasResidual;
  // Residuals ahead of the stores: C may alias the residual, so a load after
  // a store would wait for it.
  constexpr int kPerWave = (kTM * kTN + T::kWaves - 1) / T::kWaves;
  float addend[kPerWave][4];
#pragma unroll
  for (int q = 0; q < kPerWave; ++q) {
    const int t = min(wave + q * T::kWaves, kTM * kTN - 1);
    const int col = min(block_n * kBN + (t % kTN) * 16 + r16, N - 1);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = min(m0 + (t / kTN) * 16 + 4 * g + e, M - 1);
      addend[q][e] = res_mode ? epi.residual[static_cast<size_t>(row) * ldc + col] : 0.0F;
    }
  }
#pragma unroll
  for (int q = 0; q < kPerWave; ++q) {
    const int t = wave + q * T::kWaves;
    const int col = block_n * kBN + (t % kTN) * 16 + r16;
    if (t >= kTM * kTN || col >= N)
      continue;
    const f32x4 v = total(t / kTN, t % kTN);
    const float bias = bias_mode ? bf16_to_f32(epi.bias[col]) : 0.0F;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = m0 + (t / kTN) * 16 + 4 * g + e;
      if (row < M) {
        float value = v[e];
        if (bias_mode)
          value = value + bias;
        if (res_mode)
          value = value + addend[q][e];
        C[static_cast<size_t>(row) * ldc + col] = value;
      }
    }
  }
}

template <typename T, bool kSplit, bool kF16>
Status launch(const TileCall &c, hipStream_t stream) {
  constexpr size_t stage = ((kSplit ? 2 : 1) * T::kBM + T::kBN) * T::kSeg * 2;
  constexpr size_t lds = std::max<size_t>(T::kStages * stage,
                                          static_cast<size_t>(T::kWK) * T::kBM * T::kBN * 4);
  static_assert(lds <= 160 * 1024, "LDS");
  const auto kernel = gemm_tile_kernel<T, kSplit, kF16>;
  if (lds > 64 * 1024)
    EVO_TRY(hip_status(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           static_cast<int>(lds)),
                       "gemm_tile_kernel LDS opt-in"));
  const dim3 grid(ceil_div(c.M, T::kBM) * ceil_div(c.N, T::kBN), static_cast<unsigned>(c.splits));
  hipLaunchKernelGGL(kernel, grid, dim3(T::kWaves * 64), lds, stream, c.a_hi, c.a_lo, c.lda, c.W,
                     c.K, c.M, c.N, c.K / c.splits, c.C, c.c_split, c.c_hi, c.c_lo, c.ldc, c.epi);
  return launch_status("gemm_tile_kernel");
}

template <typename T> Status launch_planes(const TileCall &c, hipStream_t stream) {
  if (c.a_lo != nullptr)
    return launch<T, true, false>(c, stream);
  return c.f16 ? launch<T, false, true>(c, stream) : launch<T, false, false>(c, stream);
}

struct TileEntry {
  int bm, bn, seg;
  TileCost split, plane;  // hi + lo activation planes, one plane
};
// Least-squares fits over 5 to 8192 rows of ten (N, K), those of the 7B and 1B
// topologies among them (median error 2-6 %), each then scaled by 1.00 to 1.15
// so that the choice among the tiles is the best one: with the plain fits,
// products of a few thousand rows were up to 10 % slower than on 256 x 256
// tiles (5000 rows of 4096 x 4096, two planes: 407 us on 128 x 128, 366 there).
// Over 1060 products, with and without a workspace, the choice takes 0.4 % more
// than the fastest tile and split in the geometric mean, 21 % at worst (5 rows
// of 512 x 4096, one plane), and 4 % more than 256 x 256 at worst.
constexpr TileEntry kTiles[] = {
    {16, 16, 128, {1.91F, 1.35F, 0.013F, 2, {0.215F, 0.372F}, 7.12F}, {2.09F, 1.09F, 0.0F, 3, {0.203F, 0.302F, 0.397F}, 5.36F}},
    {16, 32, 128, {2.56F, 1.13F, 0.022F, 2, {0.298F, 0.519F}, 4.78F}, {2.14F, 1.1F, 0.013F, 2, {0.254F, 0.379F}, 5.17F}},
    {32, 32, 128, {1.83F, 2.13F, 0.125F, 1, {0.311F}, 7.32F}, {1.87F, 1.91F, 0.043F, 1, {0.275F}, 4.99F}},
    {32, 64, 128, {2.09F, 1.96F, 0.176F, 1, {0.389F}, 4.73F}, {2.26F, 1.96F, 0.083F, 1, {0.349F}, 4.58F}},
    {32, 96, 128, {2.67F, 2.29F, 0.16F, 1, {0.561F}, 4.42F}, {2.76F, 2.16F, 0.087F, 1, {0.528F}, 4.29F}},
    {64, 64, 64, {1.89F, 2.68F, 0.096F, 1, {0.326F}, 7.27F}, {2.31F, 2.54F, 0.019F, 2, {0.288F, 0.503F}, 4.61F}},
    {64, 128, 64, {2.59F, 4.18F, 0.126F, 1, {0.43F}, 4.22F, 6.66F}, {3.25F, 3.54F, 0.073F, 1, {0.358F}, 4.06F}},
    {64, 192, 64, {2.39F, 5.88F, 0.164F, 1, {0.587F}, 4.38F, 6.12F}, {3.41F, 5.12F, 0.073F, 1, {0.527F}, 3.95F}},
    {128, 128, 64, {2.07F, 6.02F, 0.19F, 1, {0.735F}, 8.57F, 6.34F}, {1.37F, 6.6F, 0.126F, 1, {0.461F}, 4.18F, 6.11F}},
    {128, 192, 64, {2.91F, 7.01F, 0.27F, 1, {1.144F}, 4.01F, 5.18F}, {3.84F, 5.9F, 0.219F, 1, {0.876F}, 3.92F}},
};
constexpr int kTileCount = static_cast<int>(sizeof(kTiles) / sizeof(kTiles[0]));
static_assert(kTileCount == kGemmTiles, "the tiles of gemm_tile()");
// The 256 x 256 tile of gemm.hip, the other candidate.
constexpr TileEntry kLargeTile = {256, 256, 32, {0.0F, 7.29F, 0.532F, 1, {1.041F}},
                                  {0.0F, 7.71F, 0.233F, 1, {0.750F}}};

float entry_us(const TileEntry &t, bool split, uint32_t M, uint32_t N, uint32_t k_part,
               uint32_t parts, float weight_bytes, float limit) {
  const TileCost &cost = split ? t.split : t.plane;
  const uint32_t down = (M + t.bm - 1) / t.bm, blocks = down * ((N + t.bn - 1) / t.bn) * parts;
  float fill_bytes = 0.0F;
  if (cost.fill > 0.0F) {
    // An XCD's resident blocks are consecutive, rows first: 32 row blocks and
    // more share no activation rows, which each block column then reads again.
    const float all = static_cast<float>(blocks);
    const float resident = std::min(32.0F * cost.slots, std::max(1.0F, all / 8.0F));
    const float shared = std::min(static_cast<float>(down), resident);
    const float rows = shared * t.bm * (split ? 2 : 1) + std::max(1.0F, resident / shared) * t.bn;
    fill_bytes = all / resident * rows * 2.0F * static_cast<float>(k_part);
  }
  return tile_us(cost, blocks, (k_part + t.seg - 1) / t.seg, weight_bytes, fill_bytes, limit);
}

}  // namespace

TileChoice choose_gemm_tile(size_t M, size_t N, size_t K, bool split, bool gated,
                            size_t large_parts, size_t workspace_bytes, bool deferred) {
  // Partial products cost their reduction: a launch that grows with the parts
  // (5 rows of 1920 x 5120, two planes: 4 parts 9.8 us, 8 parts 11.1) unless
  // the next norm sums them as it reads its rows, and their bytes at ~4 TB/s.
  const float weight_bytes = 2.0F * static_cast<float>(N) * static_cast<float>(K);
  const float part_us = static_cast<float>(M) * static_cast<float>(N) * 1.0e-6F;
  auto reduction = [&](size_t parts) {
    return parts == 1 ? 0.0F
                      : (deferred ? 0.0F : 2.0F + 0.3F * static_cast<float>(parts)) +
                            static_cast<float>(parts) * part_us;
  };
  const auto m = static_cast<uint32_t>(M), n = static_cast<uint32_t>(N);
  TileChoice best;
  float best_us = entry_us(kLargeTile, split, m, n, static_cast<uint32_t>(K / large_parts),
                           static_cast<uint32_t>(large_parts), weight_bytes, INFINITY) +
                  reduction(large_parts);
  const size_t plane_bytes = M * N * sizeof(float);
  const bool splittable = !gated && N % 4 == 0;
  for (size_t parts = 1; parts <= 8; parts *= 2) {
    if (K % (32 * parts) != 0 || (parts > 1 && (!splittable || parts * plane_bytes > workspace_bytes)))
      break;
    const auto k_part = static_cast<uint32_t>(K / parts);
    const float reduce_us = reduction(parts);
    for (int t = 0; t < kTileCount; ++t) {
      if (gated && kTiles[t].bn % 32 != 0)
        continue;  // a gated tile pairs whole 16-column tiles
      if (k_part < static_cast<uint32_t>((parts > 1 ? 4 : 1) * kTiles[t].seg))
        continue;
      const float us = entry_us(kTiles[t], split, m, n, k_part, static_cast<uint32_t>(parts),
                                weight_bytes, best_us - reduce_us) +
                       reduce_us;
      if (us < best_us) {
        best_us = us;
        best = TileChoice{t, static_cast<int>(parts)};
      }
    }
  }
  return best;
}

Status gemm_tile(int tile, const TileCall &call, hipStream_t stream) {
  // The shapes of kTiles, in its order.
  switch (tile) {
  case 0: return launch_planes<TileShape<16, 16, 128, 4, 1, 1, 6>>(call, stream);
  case 1: return launch_planes<TileShape<16, 32, 128, 4, 1, 1, 5>>(call, stream);
  case 2: return launch_planes<TileShape<32, 32, 128, 4, 2, 1, 6>>(call, stream);
  case 3: return launch_planes<TileShape<32, 64, 128, 4, 2, 1, 5>>(call, stream);
  case 4: return launch_planes<TileShape<32, 96, 128, 4, 2, 1, 4>>(call, stream);
  case 5: return launch_planes<TileShape<64, 64, 64, 2, 4, 1, 4>>(call, stream);
  case 6: return launch_planes<TileShape<64, 128, 64, 2, 4, 1, 4>>(call, stream);
  case 7: return launch_planes<TileShape<64, 192, 64, 2, 4, 1, 4>>(call, stream);
  case 8: return launch_planes<TileShape<128, 128, 64, 2, 4, 1, 3>>(call, stream);
  case 9: return launch_planes<TileShape<128, 192, 64, 1, 4, 2, 2>>(call, stream);
  default: return {ErrorCode::kInternal, "gemm_tile: unknown tile"};
  }
}

}  // namespace evo::hip
