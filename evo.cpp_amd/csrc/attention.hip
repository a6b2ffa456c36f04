// SPDX-License-Identifier: Apache-2.0
// Attention block of StripedHyena2 on gfx950 (prefill; single-query decode).
//
// qkv_rope: splits the Wqkv projection (head-major `column_split` layout
// [h][q,k,v][d], or component-major [q,k,v][h][d]), applies GPT-NeoX
// half-pair RoPE at position (prefix + row) / rope_scale and writes Q and the
// appended K rows as split BF16 planes (hi = bf16(x), lo = bf16(x - hi)).
// v_transpose appends V to the transposed value cache V^T [W][capacity]
// (row h*d_head + d), keys permuted inside every 16-key block by swapping
// bits 2 and 3 of the position, the order in which one MFMA lane holds the
// probabilities of a 16-key step (see below).
// Reference: evo.cpp `src/cpu/model.cpp:455-509`.
//
// causal_attention: softmax(q.k / sqrt(d)) v over keys [0, position].
// Reference semantics: `src/cpu/model.cpp:510-544` (full softmax; the online
// form below equals it up to F32 rounding).
//
// MFMA kernel (head_dim 32/64/128): one block = 8 or 4 waves x 32 queries of
// one head, over all of its keys or, with a workspace, a part of them
// (plan_flash; flash_combine_kernel joins the parts). K [32 keys][d] and V^T
// [d][32 keys] tiles of both planes are DMA'd (global_load_lds) into
// XOR-swizzled LDS, double buffered, so the next tile streams in while this
// one computes. 8192 x 4096 and 4096 x 4096 on a prefix of 28672 take 1350 and
// 4850 us (64-key tiles, per-lane DMA addresses and fragment reads right
// before their MFMAs: 1530 and 5150); the matrix cores run at 1.3 PFLOP/s of
// three-pass work there, near what random operands sustain. Each wave computes
// S^T = K Q^T (keys x queries) with v_mfma_f32_32x32x16_bf16, so every lane
// owns one query: the running max and sum stay in-lane (plus one exchange
// with the lane holding the other half of the keys), and P^T is already in
// the B-operand layout of O^T += V^T P^T. Products use three BF16 passes
// (hi*hi + hi*lo + lo*hi), about 16 significant bits per operand, with F32
// accumulation; the exponential is exp2 of log2(e)-prescaled scores.
// head_dim 16 uses a VALU kernel (four lanes per query).
#include "common.hpp"
#include "ops.hpp"

#include <algorithm>
#include <cmath>

namespace evo::hip {

// FP16-plane attention output without a per-value range check: the outputs
// are convex combinations of V rows, whose range qkv_rope checks as they
// enter the cache.
struct F16Plane {
  uint16_t *out;
};
__device__ inline void put(const F16Plane &o, size_t i, float v) {
  o.out[i] = f32_to_f16_sat(v);
}

namespace {

__device__ inline void put_split(uint16_t *hi, uint16_t *lo, size_t i, float v) {
  const uint16_t h = f32_to_bf16(v);
  hi[i] = h;
  lo[i] = f32_to_bf16(v - bf16_to_f32(h));
}

__device__ inline float get_split(const uint16_t *hi, const uint16_t *lo, size_t i) {
  return bf16_to_f32(hi[i]) + bf16_to_f32(lo[i]);
}

// hi + lo of 8 consecutive elements.
__device__ inline void split_floats(const uint4 &hi, const uint4 &lo, float (&v)[8]) {
  const uint32_t h[4] = {hi.x, hi.y, hi.z, hi.w}, l[4] = {lo.x, lo.y, lo.z, lo.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __builtin_bit_cast(float, h[i] << 16) + __builtin_bit_cast(float, l[i] << 16);
    v[2 * i + 1] = __builtin_bit_cast(float, h[i] & 0xffff0000U) +
                   __builtin_bit_cast(float, l[i] & 0xffff0000U);
  }
}

// Position of key `pos` inside the transposed value cache.
__host__ __device__ inline size_t vt_column(size_t pos) {
  return (pos & ~static_cast<size_t>(15)) | (pos & 3) | ((pos & 4) << 1) | ((pos & 8) >> 1);
}

__device__ inline size_t qkv_column(int column_split, size_t width, size_t head,
                                    size_t head_dim, size_t component, size_t dim) {
  return column_split ? head * 3 * head_dim + component * head_dim + dim
                      : component * width + head * head_dim + dim;
}

// Consecutive split-BF16 elements: kVec planes' words in one store each.
template <int kVec>
__device__ inline void put_split_vec(uint16_t *hi, uint16_t *lo, const float (&v)[kVec]) {
  if constexpr (kVec == 1) {
    put_split(hi, lo, 0, v[0]);
  } else {
    uint16_t h[kVec], l[kVec];
#pragma unroll
    for (int e = 0; e < kVec; ++e) {
      h[e] = f32_to_bf16(v[e]);
      l[e] = f32_to_bf16(v[e] - bf16_to_f32(h[e]));
    }
    *reinterpret_cast<uint2 *>(hi) = __builtin_bit_cast(uint2, h);
    *reinterpret_cast<uint2 *>(lo) = __builtin_bit_cast(uint2, l);
  }
}
template <int kVec>
__device__ inline void load_floats(const float *src, float (&v)[kVec]) {
  if constexpr (kVec == 1) {
    v[0] = src[0];
  } else {
    const float4 f = *reinterpret_cast<const float4 *>(src);
    v[0] = f.x;
    v[1] = f.y;
    v[2] = f.z;
    v[3] = f.w;
  }
}

struct QkvAppend {
  const float *projected;
  size_t rows, width, heads;
  int half;  // rotation pairs per head
  int column_split;
  const float *inv_freq;
  float rope_scale;
  size_t prefix;
  uint16_t *q;
  size_t q_plane;
  uint16_t *k_cache, *vt_cache;
  size_t cache_plane, capacity;
  int *range_flag;
  unsigned value_blocks, row_parts;
};

// Rotated q and k of one row (or, with row_parts > 1, of a part of its
// heads): a thread owns kVec rotation pairs of every head_step-th head, so
// their cosines and sines are evaluated once.
template <int kVec>
__device__ inline void rotate_row(const QkvAppend &a, size_t row, int part) {
  const size_t head_dim = 2 * static_cast<size_t>(a.half);
  const int lanes = a.half / kVec;  // threads per head
  const int head_step = 256 / lanes;
  const int pair = static_cast<int>(threadIdx.x) % lanes * kVec;
  const float *src = a.projected + row * a.width * 3;
  const float position = static_cast<float>(a.prefix + row) / a.rope_scale;
  float cosine[kVec], sine[kVec];
#pragma unroll
  for (int e = 0; e < kVec; ++e) {
    const float angle = position * a.inv_freq[pair + e];
    cosine[e] = cosf(angle);
    sine[e] = sinf(angle);
  }
  for (size_t head = threadIdx.x / lanes + static_cast<size_t>(part) * head_step; head < a.heads;
       head += static_cast<size_t>(head_step) * a.row_parts) {
#pragma unroll
    for (int component = 0; component < 2; ++component) {
      float first[kVec], second[kVec], x[kVec], y[kVec];
      load_floats(src + qkv_column(a.column_split, a.width, head, head_dim, component, pair),
                  first);
      load_floats(
          src + qkv_column(a.column_split, a.width, head, head_dim, component, a.half + pair),
          second);
#pragma unroll
      for (int e = 0; e < kVec; ++e) {
        x[e] = first[e] * cosine[e] - second[e] * sine[e];
        y[e] = second[e] * cosine[e] + first[e] * sine[e];
      }
      const size_t at = (component == 0 ? row : a.prefix + row) * a.width + head * head_dim + pair;
      uint16_t *hi = (component == 0 ? a.q : a.k_cache) + at;
      uint16_t *lo = hi + (component == 0 ? a.q_plane : a.cache_plane);
      put_split_vec(hi, lo, x);
      put_split_vec(hi + a.half, lo + a.half, y);
    }
  }
}

// V rows [rows, W] of the projection -> V^T planes at positions prefix..:
// a 64-position x 64-channel tile is read row-wise, transposed through LDS
// and written position-contiguous.
template <int kVec>
__device__ inline void transpose_values(const QkvAppend &a, size_t r0, size_t c0,
                                        float (*tile)[65]) {
  constexpr int kLanes = 64 / kVec, kStep = 256 / kLanes;  // lanes per row, rows per pass
  const int tid = threadIdx.x;
  const size_t head_dim = 2 * static_cast<size_t>(a.half);
  const int offset = tid % kLanes * kVec;
  const size_t channel = c0 + offset;
  const float *src = a.projected + qkv_column(a.column_split, a.width, channel / head_dim,
                                              head_dim, 2, channel % head_dim);
  bool out_of_range = false;
#pragma unroll
  for (int i0 = 0; i0 < 64; i0 += kStep) {
    const int i = i0 + tid / kLanes;
    float value[kVec] = {};
    if (r0 + i < a.rows && channel < a.width)
      load_floats(src + (r0 + i) * a.width * 3, value);
#pragma unroll
    for (int e = 0; e < kVec; ++e) {
      out_of_range |= !(__builtin_fabsf(value[e]) <= 65504.0F);
      tile[offset + e][i] = value[e];
    }
  }
  if (a.range_flag != nullptr && out_of_range)
    atomicOr(a.range_flag, kFlagF16Range);
  __syncthreads();
  if (a.prefix % 16 == 0 && r0 + 64 <= a.rows && c0 + 64 <= a.width) {
    // Whole tile from a 16-aligned position: its 64 V^T columns per channel
    // are [prefix + r0, +64) in the permuted order; each lane packs 8 of
    // them (column j holds row vt_column(j), the permutation being its own
    // inverse) into one 16-byte store per plane.
    uint16_t *base = a.vt_cache + a.prefix + r0;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int idx = tid + 256 * k, i = idx >> 3, unit = idx & 7;
      uint32_t hi[4], lo[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float v0 = tile[i][vt_column(8 * unit + e)];
        const float v1 = tile[i][vt_column(8 * unit + e + 1)];
        const uint16_t h0 = f32_to_bf16(v0), h1 = f32_to_bf16(v1);
        hi[e / 2] = h0 | (static_cast<uint32_t>(h1) << 16);
        lo[e / 2] = f32_to_bf16(v0 - bf16_to_f32(h0)) |
                    (static_cast<uint32_t>(f32_to_bf16(v1 - bf16_to_f32(h1))) << 16);
      }
      const size_t at = (c0 + i) * a.capacity + 8 * unit;
      *reinterpret_cast<uint4 *>(base + at) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
      *reinterpret_cast<uint4 *>(base + a.cache_plane + at) =
          make_uint4(lo[0], lo[1], lo[2], lo[3]);
    }
    return;
  }
  const int rows_here = static_cast<int>(min(static_cast<size_t>(64), a.rows - r0));
  const int channels = static_cast<int>(min(static_cast<size_t>(64), a.width - c0));
  // A few rows (the decode step): lanes on the channels, else on the rows.
  for (int j = tid; j < rows_here * channels; j += 256) {
    const int i = j / rows_here, row = j % rows_here;
    put_split(a.vt_cache, a.vt_cache + a.cache_plane,
              (c0 + i) * a.capacity + vt_column(a.prefix + r0 + row), tile[i][row]);
  }
}

// q, k and v of a projection in one launch: the first value_blocks blocks
// write V^T tiles, the others rotate rows. Bound by bytes (F32 in, two
// planes out): 1500 x 1920 takes 18 us, one decode row of 4096 5.0 (a launch
// each, one scalar pair or channel per thread: 26.6 and 13.8).
template <int kVec>
__global__ __launch_bounds__(256) void append_qkv_kernel(const QkvAppend a) {
  __shared__ float tile[64][65];
  const unsigned b = blockIdx.x;
  if (b < a.value_blocks) {
    const unsigned columns = static_cast<unsigned>((a.width + 63) / 64);
    transpose_values<kVec>(a, b / columns * 64ULL, b % columns * 64ULL, tile);
  } else {
    const unsigned r = b - a.value_blocks;
    rotate_row<kVec>(a, r / a.row_parts, static_cast<int>(r % a.row_parts));
  }
}

// ------------------------------------------------------------ MFMA kernel
constexpr int kKeys = 64;            // cache capacity granule
constexpr int kQueriesPerWave = 32;
constexpr int kTileKeys = 32;        // keys of a K/V tile

// Swizzle of a row of kUnits 16-byte units: 8 consecutive rows read at one
// logical unit hit 8 distinct 16-byte bank groups.
template <int kUnits>
__device__ inline int swizzle(int row, int unit) {
  return unit ^ ((row * kUnits / 16) & (kUnits - 1));
}

template <int kD, int kWaves>
struct FlashShape {
  static constexpr int kQueries = kWaves * kQueriesPerWave;
  static constexpr int kKUnits = kD / 8;             // 16-byte units per K row
  static constexpr int kVUnits = kTileKeys / 8;      // and per V^T row
  static constexpr int kPlane = kTileKeys * kD;      // BF16 per K or V^T plane
  static constexpr int kStage = 4 * kPlane;          // {K hi, K lo, V hi, V lo}
  static constexpr size_t kLdsBytes = 2 * kStage * sizeof(uint16_t);
  static constexpr int kChunksPerPlane = kPlane / 512;  // 1 KB chunks
  static constexpr int kDmaPerWave = 4 * kChunksPerPlane / kWaves;
  static_assert(4 * kChunksPerPlane % kWaves == 0, "DMA split");
};

// Key split of a launch: query block qb of T key tiles runs as
// ceil(T / chunk_tiles) blocks over equal parts of its tiles (at most
// max_chunks), each leaving its unnormalised output, running maximum (log2
// domain) and sum in `part` for flash_combine_kernel; a query block of one
// part writes its output itself. max_chunks == 1: no split.
struct KeySplit {
  uint32_t chunk_tiles, max_chunks;
  float *part;  // [heads][query blocks][max_chunks][kQueries][kD + 2]
};
__device__ inline uint32_t key_chunks(const KeySplit &split, uint32_t tiles) {
  return split.max_chunks == 1 ? 1 : (tiles + split.chunk_tiles - 1) / split.chunk_tiles;
}
__device__ inline uint32_t key_tiles(size_t prefix, size_t rows, size_t block_row, int queries) {
  const size_t last = min(rows, block_row + queries) - 1;
  return static_cast<uint32_t>((prefix + last) / kTileKeys + 1);
}

// Order of kGroups groups of {two LDS fragment reads, three MFMAs on them}
// between the surrounding scheduling barriers: the reads run kAhead groups
// ahead of the MFMAs that use them. (Left to itself the compiler reads each
// pair right before its MFMAs and waits out the LDS latency every time.)
template <int kGroups, int kAhead, int kReadGroups> __device__ inline void schedule_reads_ahead() {
  if (kAhead > 0)
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAhead, 0);
#pragma unroll
  for (int i = 0; i < kGroups; ++i) {
    if (i + kAhead < kReadGroups)
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
}

// kWide: V^T row offsets within a DMA need more than 32 bits (2^27 positions).
template <int kD, typename O, int kWaves, bool kWide>
__global__ __launch_bounds__(kWaves * 64, 2) void flash_attention_kernel(
    const uint16_t *__restrict__ q, size_t q_plane, const uint16_t *__restrict__ k_cache,
    const uint16_t *__restrict__ vt_cache, size_t cache_plane, size_t capacity, size_t rows,
    size_t prefix, size_t heads, const KeySplit split, O out) {
  using Shape = FlashShape<kD, kWaves>;
  constexpr int kDSteps = kD / 16;  // K-steps of S^T over head_dim
  constexpr int kDTiles = kD / 32;  // 32-row tiles of O^T
  extern __shared__ __attribute__((aligned(16))) uint16_t flash_lds[];

  const size_t width = heads * kD;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, col = lane & 31;
  // Block -> (head, query block, key chunk): heaviest (latest) query blocks
  // first; with heads % 8 == 0 the blocks of a head share an XCD (blocks are
  // dealt to the 8 XCDs round-robin), so its K/V tiles are reused from one L2.
  const size_t query_blocks = (rows + Shape::kQueries - 1) / Shape::kQueries;
  const size_t b = blockIdx.x;
  size_t head, rest;
  if (heads % 8 == 0) {
    const size_t per_xcd = heads / 8, idx = b / 8;
    head = (b % 8) + 8 * (idx % per_xcd);
    rest = idx / per_xcd;
  } else {
    head = b % heads;
    rest = b / heads;
  }
  const size_t qb = query_blocks - 1 - rest / split.max_chunks;
  const uint32_t chunk = static_cast<uint32_t>(rest % split.max_chunks);
  const size_t block_row = qb * Shape::kQueries;
  const uint32_t all_tiles = key_tiles(prefix, rows, block_row, Shape::kQueries);
  const uint32_t chunks = key_chunks(split, all_tiles);
  if (chunk >= chunks)
    return;
  const uint32_t first_tile = static_cast<uint32_t>(static_cast<uint64_t>(all_tiles) * chunk / chunks);
  const uint32_t end_tile =
      static_cast<uint32_t>(static_cast<uint64_t>(all_tiles) * (chunk + 1) / chunks);
  const size_t row = block_row + wave * kQueriesPerWave + col;  // this lane's query
  const bool active = row < rows;
  // exp(x * scale) = exp2(x * scale * log2(e))
  const float scale2 = 1.4426950408889634F / sqrtf(static_cast<float>(kD));

  // Q^T operand fragments: for d-step s, 8 consecutive dims s*16 + half*8.
  bf16x8 qh[kDSteps], ql[kDSteps];
#pragma unroll
  for (int s = 0; s < kDSteps; ++s) {
    const size_t base = (active ? row : 0) * width + head * kD + s * 16 + half * 8;
    qh[s] = *reinterpret_cast<const bf16x8 *>(q + base);
    ql[s] = *reinterpret_cast<const bf16x8 *>(q + q_plane + base);
    if (!active) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        qh[s][e] = static_cast<__bf16>(0.0F);
        ql[s][e] = static_cast<__bf16>(0.0F);
      }
    }
  }

  // DMA op g of this wave: part g / kChunksPerPlane of {K hi, K lo, V hi, V
  // lo}, 1 KB chunk g % kChunksPerPlane of that plane: a wave-uniform base
  // that advances with the tile, a fixed 32-bit byte offset per lane and a
  // wave-uniform LDS address (per-lane 64-bit sources and generic LDS
  // pointers cost ~10 instructions per DMA, ahead of each tile's first MFMA).
  const char *base[Shape::kDmaPerWave];
  uint32_t offset[Shape::kDmaPerWave];
#pragma unroll
  for (int i = 0; i < Shape::kDmaPerWave; ++i) {
    const int g = wave * Shape::kDmaPerWave + i;
    const int part = g / Shape::kChunksPerPlane, first = (g % Shape::kChunksPerPlane) * 64;
    const size_t plane = (part & 1) != 0 ? cache_plane : 0;
    if (part < 2) {
      const int key = (first + lane) / Shape::kKUnits;
      const int unit = swizzle<Shape::kKUnits>(key, (first + lane) % Shape::kKUnits);
      base[i] = reinterpret_cast<const char *>(k_cache + plane + head * kD);
      offset[i] = static_cast<uint32_t>(key * width + unit * 8) * 2;
    } else {
      // 64 lanes cover 16 rows of V^T: the first one's goes into the base.
      const int d = (first + lane) / Shape::kVUnits, d0 = first / Shape::kVUnits;
      const int unit = swizzle<Shape::kVUnits>(d, lane % Shape::kVUnits);
      base[i] = reinterpret_cast<const char *>(vt_cache + plane + (head * kD + d0) * capacity);
      offset[i] = static_cast<uint32_t>((d - d0) * capacity + unit * 8) * 2;
    }
  }
  const unsigned lds = lds_address(flash_lds);
  auto issue = [&](uint32_t tile) {
    const size_t k0 = static_cast<size_t>(tile) * kTileKeys;
#pragma unroll
    for (int i = 0; i < Shape::kDmaPerWave; ++i) {
      const bool is_k = (wave * Shape::kDmaPerWave + i) / Shape::kChunksPerPlane < 2;
      const unsigned to = wave * Shape::kDmaPerWave * 1024 + (tile & 1) * (Shape::kStage * 2) +
                          i * 1024;
      const char *from = base[i] + (is_k ? k0 * width : k0) * 2;
      if (kWide && !is_k) {
        const size_t down = (lane / Shape::kVUnits) * capacity * 2;
        dma16(from + down + (offset[i] - static_cast<uint32_t>(down)), flash_lds + to / 2);
      } else {
        dma16_at(from, offset[i], lds + to);
      }
    }
  };

  f32x16 o_acc[kDTiles];
#pragma unroll
  for (int t = 0; t < kDTiles; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e)
      o_acc[t][e] = 0.0F;
  float running_max = -INFINITY, partial_sum = 0.0F;

  // Lowest position of the wave's queries, and whether it has any.
  const size_t wave_first = prefix + block_row + wave * kQueriesPerWave;
  const bool wave_rows = block_row + wave * kQueriesPerWave < rows;
  issue(first_tile);
  for (uint32_t tile = first_tile; tile < end_tile; ++tile) {
    // This wave's DMA of the tile (the only one in flight), then one
    // barrier: every wave's DMA of the tile has landed and every wave has
    // left buffer (tile+1)&1 (tile-1's), which the next DMA overwrites.
    wait_dma<0>();
    __syncthreads();
    if (tile + 1 < end_tile)
      issue(tile + 1);
    const size_t k0 = static_cast<size_t>(tile) * kTileKeys;
    // Every key of the tile lies beyond every query of the wave.
    if (!wave_rows || k0 > wave_first + (kQueriesPerWave - 1))
      continue;
    const uint16_t *stage = flash_lds + (tile & 1) * Shape::kStage;
    const uint16_t *k_hi = stage, *k_lo = stage + Shape::kPlane;
    const uint16_t *v_hi = stage + 2 * Shape::kPlane, *v_lo = v_hi + Shape::kPlane;

    // S^T: entry e holds key (e/4)*8 + half*4 + e%4 of the tile for query col.
    f32x16 st;
#pragma unroll
    for (int e = 0; e < 16; ++e)
      st[e] = 0.0F;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < kDSteps; ++s) {
      const int off = (col * Shape::kKUnits + swizzle<Shape::kKUnits>(col, 2 * s + half)) * 8;
      const bf16x8 kh = *reinterpret_cast<const bf16x8 *>(k_hi + off);
      const bf16x8 kl = *reinterpret_cast<const bf16x8 *>(k_lo + off);
      st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kh, qh[s], st, 0, 0, 0);
      st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kh, ql[s], st, 0, 0, 0);
      st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kl, qh[s], st, 0, 0, 0);
    }
    schedule_reads_ahead<kDSteps, kDSteps < 2 ? kDSteps : 2, kDSteps>();
    // Causal mask on the diagonal tiles, tile maximum (log2 domain: the
    // scale is positive, so it commutes with the maximum).
    if (k0 + kTileKeys - 1 > wave_first) {
      // Keys from the tile's first up to this query's position.
      const int visible = static_cast<int>(wave_first - k0) + col;
#pragma unroll
      for (int e = 0; e < 16; ++e)
        st[e] = (e >> 2) * 8 + half * 4 + (e & 3) <= visible ? st[e] : -INFINITY;
    }
    auto read_v = [&](int kk, int t, bf16x8 &vh, bf16x8 &vl) {
      const int d = t * 32 + col;
      const int off = (d * Shape::kVUnits + swizzle<Shape::kVUnits>(d, 2 * kk + half)) * 8;
      vh = *reinterpret_cast<const bf16x8 *>(v_hi + off);
      vl = *reinterpret_cast<const bf16x8 *>(v_lo + off);
    };
    // The first V^T fragments arrive under the softmax.
    bf16x8 vh, vl;
    read_v(0, 0, vh, vl);
    float tile_max = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; ++e)
      tile_max = fmaxf(tile_max, st[e]);
    tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32, 64)) * scale2;
    const float new_max = fmaxf(running_max, tile_max);
    if (__any(new_max != running_max)) {
      // A query with no visible key yet keeps new_max = -inf: nothing to scale.
      const float correction =
          new_max == -INFINITY ? 1.0F : __builtin_amdgcn_exp2f(running_max - new_max);
      partial_sum *= correction;
#pragma unroll
      for (int t = 0; t < kDTiles; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          o_acc[t][e] *= correction;
      running_max = new_max;
    }
    const float base_max = new_max == -INFINITY ? 0.0F : new_max;
    // P = exp2(S * scale - max) as B operands; with the permuted V^T key
    // order, the 8 entries e0..e0+7 of this lane are the 8 consecutive V^T
    // columns of 16-key step kk at half*8.
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8 ph, pl;
#pragma unroll
      for (int slot = 0; slot < 8; ++slot) {
        const float p = __builtin_amdgcn_exp2f(fmaf(st[kk * 8 + slot], scale2, -base_max));
        partial_sum += p;
        const __bf16 h = static_cast<__bf16>(p);
        ph[slot] = h;
        pl[slot] = static_cast<__bf16>(p - static_cast<float>(h));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < kDTiles; ++t) {
        bf16x8 next_h = vh, next_l = vl;
        if (t + 1 < kDTiles)
          read_v(kk, t + 1, next_h, next_l);
        else if (kk == 0)
          read_v(1, 0, next_h, next_l);
        o_acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vh, ph, o_acc[t], 0, 0, 0);
        o_acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vh, pl, o_acc[t], 0, 0, 0);
        o_acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vl, ph, o_acc[t], 0, 0, 0);
        vh = next_h;
        vl = next_l;
      }
      if (kk == 0)
        schedule_reads_ahead<kDTiles, 0, kDTiles>();
      else
        schedule_reads_ahead<kDTiles, 0, kDTiles - 1>();
    }
  }
  const float total = partial_sum + __shfl_xor(partial_sum, 32, 64);
  if (!active)
    return;
  // O^T entry e of tile t: d = t*32 + (e/4)*8 + half*4 + e%4, query = col.
  if (chunks > 1) {
    float *dst = split.part + (((head * query_blocks + qb) * split.max_chunks + chunk) *
                                   Shape::kQueries + wave * kQueriesPerWave + col) * (kD + 2);
    if (half == 0) {
      dst[0] = running_max;
      dst[1] = total;
    }
#pragma unroll
    for (int t = 0; t < kDTiles; ++t)
#pragma unroll
      for (int e = 0; e < 16; e += 2)
        *reinterpret_cast<float2 *>(dst + 2 + t * 32 + (e >> 2) * 8 + half * 4 + (e & 3)) =
            make_float2(o_acc[t][e], o_acc[t][e + 1]);
    return;
  }
#pragma unroll
  for (int t = 0; t < kDTiles; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int d = t * 32 + (e >> 2) * 8 + half * 4 + (e & 3);
      put(out, row * width + head * kD + d, o_acc[t][e] / total);
    }
}

// Rows of split query blocks: the chunks rescaled to their common maximum and
// summed in chunk order. One wave per (row, head), two dims per lane (kD / 2
// lanes).
template <int kD, typename O, int kWaves>
__global__ __launch_bounds__(256) void flash_combine_kernel(size_t rows, size_t prefix,
                                                            size_t heads, const KeySplit split,
                                                            O out) {
  using Shape = FlashShape<kD, kWaves>;
  const size_t index = blockIdx.x * 4ULL + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const size_t row = index / heads, head = index % heads;
  if (row >= rows || lane >= kD / 2)
    return;
  const size_t query_blocks = (rows + Shape::kQueries - 1) / Shape::kQueries;
  const size_t qb = row / Shape::kQueries;
  const uint32_t chunks =
      key_chunks(split, key_tiles(prefix, rows, qb * Shape::kQueries, Shape::kQueries));
  if (chunks == 1)
    return;
  const float *src = split.part + ((head * query_blocks + qb) * split.max_chunks * Shape::kQueries +
                                   row % Shape::kQueries) * (kD + 2);
  constexpr size_t kStep = Shape::kQueries * (kD + 2);  // chunk to chunk
  float top = -INFINITY;
  for (uint32_t c = 0; c < chunks; ++c)
    top = fmaxf(top, src[c * kStep]);
  float sum = 0.0F, o0 = 0.0F, o1 = 0.0F;
  for (uint32_t c = 0; c < chunks; ++c) {
    // (A chunk whose keys all lie beyond the query has maximum -inf, sum 0.)
    const float m = src[c * kStep];
    const float scale = m == -INFINITY ? 0.0F : __builtin_amdgcn_exp2f(m - top);
    const float2 o = *reinterpret_cast<const float2 *>(src + c * kStep + 2 + 2 * lane);
    sum = fmaf(src[c * kStep + 1], scale, sum);
    o0 = fmaf(o.x, scale, o0);
    o1 = fmaf(o.y, scale, o1);
  }
  const size_t at = row * heads * kD + head * kD + 2 * lane;
  put(out, at, o0 / sum);
  put(out, at + 1, o1 / sum);
}

// ------------------------------------------------------------ VALU kernel
template <int kDim, typename O>  // head_dim, output type
__global__ __launch_bounds__(256) void attention_kernel(
    const uint16_t *__restrict__ q, size_t q_plane, const uint16_t *__restrict__ k_cache,
    const uint16_t *__restrict__ v_cache, size_t cache_plane, size_t capacity, size_t rows,
    size_t prefix, size_t heads, O out) {
  constexpr int kQ = 64, kTile = 64, kPart = kDim / 4;
  __shared__ float k_s[kTile * kDim];
  __shared__ float v_s[kTile * kDim];
  const size_t width = heads * kDim;
  const int tid = threadIdx.x;
  const int qi = tid >> 2, part = tid & 3;
  const size_t head = blockIdx.y;
  const size_t row = blockIdx.x * static_cast<size_t>(kQ) + qi;
  const bool active = row < rows;
  const size_t position = prefix + row;
  const float scale = 1.0F / sqrtf(static_cast<float>(kDim));
  float qv[kPart], acc[kPart];
#pragma unroll
  for (int d = 0; d < kPart; ++d) {
    qv[d] = active ? get_split(q, q + q_plane, row * width + head * kDim + part * kPart + d)
                   : 0.0F;
    acc[d] = 0.0F;
  }
  float running_max = -INFINITY, denominator = 0.0F;
  const size_t last_row = min(rows, blockIdx.x * static_cast<size_t>(kQ) + kQ) - 1;
  const size_t keys_needed = prefix + last_row + 1;
  for (size_t k0 = 0; k0 < keys_needed; k0 += kTile) {
    __syncthreads();
    for (int i = tid; i < kTile * kDim; i += 256) {
      const int key = i / kDim, d = i % kDim;
      const size_t g = (k0 + key) * width + head * kDim + d;
      const bool ok = k0 + key < keys_needed;
      k_s[i] = ok ? get_split(k_cache, k_cache + cache_plane, g) : 0.0F;
      v_s[i] = ok ? get_split(v_cache, v_cache + cache_plane,
                              (head * kDim + d) * capacity + vt_column(k0 + key))
                  : 0.0F;
    }
    __syncthreads();
    float scores[kTile];
    float tile_max = -INFINITY;
#pragma unroll
    for (int j = 0; j < kTile; ++j) {
      float dot = 0.0F;
#pragma unroll
      for (int d = 0; d < kPart; ++d)
        dot += qv[d] * k_s[j * kDim + part * kPart + d];
      dot += __shfl_xor(dot, 1, 64);
      dot += __shfl_xor(dot, 2, 64);
      scores[j] = k0 + j <= position ? dot * scale : -INFINITY;
      tile_max = fmaxf(tile_max, scores[j]);
    }
    if (tile_max == -INFINITY)
      continue;  // every key of this tile lies beyond this query
    const float new_max = fmaxf(running_max, tile_max);
    const float correction = expf(running_max - new_max);
    denominator *= correction;
#pragma unroll
    for (int d = 0; d < kPart; ++d)
      acc[d] *= correction;
    running_max = new_max;
#pragma unroll
    for (int j = 0; j < kTile; ++j) {
      const float p = expf(scores[j] - new_max);
      denominator += p;
#pragma unroll
      for (int d = 0; d < kPart; ++d)
        acc[d] += p * v_s[j * kDim + part * kPart + d];
    }
  }
  if (active) {
#pragma unroll
    for (int d = 0; d < kPart; ++d)
      put(out, row * width + head * kDim + part * kPart + d, acc[d] / denominator);
  }
}

// Block size and key split of a launch: the plan of least fitted time (us,
// head_dim 128, 130 (rows, prefix, heads) from 5 x 0 to 4096 x 28000; the
// plan it picks is within 6 % of the fastest one there). Blocks of 8 waves
// (256 queries, one per CU) need 1.67 us per 32-key tile of the longest one,
// blocks of 4 waves (128 queries) 1.36, or 2.11 when two share a CU; a full
// chip 2.63 / 1.60 us per tile and CU; keys and values come from HBM at
// 5 TB/s; a split costs its second launch and its partials' bytes. Few
// queries on a long prefix leave most CUs idle without a split (64 rows,
// prefix 8000, 32 heads: 390 -> 59 us), and so do the last query blocks of a
// prompt (1500 rows, 15 heads: 94 -> 52 us); chunks of a few thousand rows
// and more fill the chip and stay unsplit. head_dim 64 and 32 have shorter
// tiles and no fit of their own: the plan splits a little early there (611
// rows, 64 heads of 32: 34 us, 29 unsplit).
struct FlashPlan {
  int waves;
  uint32_t chunk_tiles, max_chunks;
};
double flash_plan_us(size_t rows, size_t prefix, size_t heads, size_t head_dim,
                     const FlashPlan &plan, size_t *part_bytes) {
  const size_t queries = static_cast<size_t>(plan.waves) * kQueriesPerWave;
  const size_t query_blocks = (rows + queries - 1) / queries;
  double total = 0.0, longest = 0.0, items = 0.0, parts = 0.0;
  for (size_t qb = 0; qb < query_blocks; ++qb) {
    const size_t last = std::min(rows, (qb + 1) * queries) - 1;
    const double tiles = static_cast<double>((prefix + last) / kTileKeys + 1);
    const double chunks = plan.max_chunks == 1 ? 1.0 : std::ceil(tiles / plan.chunk_tiles);
    total += tiles;
    items += chunks;
    longest = std::max(longest, std::ceil(tiles / chunks));
    parts += chunks > 1.0 ? chunks : 0.0;
  }
  const double heads_d = static_cast<double>(heads);
  total *= heads_d;
  items *= heads_d;
  const double row_bytes = static_cast<double>((head_dim + 2) * sizeof(float));
  *part_bytes = query_blocks * heads * plan.max_chunks * queries * (head_dim + 2) * sizeof(float);
  double us, fill;
  if (plan.waves == 8) {
    us = longest * 1.67;
    fill = total / 256.0 * 2.63 + (items > 256.0 ? 0.31 * us : 0.0);
  } else {
    us = longest * (items > 256.0 ? 2.11 : 1.36);
    fill = total / 256.0 * 1.60 + (items > 512.0 ? 0.08 * longest : 0.0);
  }
  const double key_bytes = 8.0 * static_cast<double>(prefix + rows) * heads_d * head_dim;
  us = std::max({us, fill, key_bytes / 5.0e6}) + 6.0;
  if (plan.max_chunks > 1)
    us += 2.7 + 2.0 * parts * heads_d * queries * row_bytes / 4.3e6;
  return us;
}
FlashPlan plan_flash(size_t rows, size_t prefix, size_t heads, size_t head_dim,
                     size_t workspace_bytes) {
  FlashPlan best{8, 0, 1};
  size_t part_bytes = 0;
  double best_us = flash_plan_us(rows, prefix, heads, head_dim, best, &part_bytes);
  auto consider = [&](const FlashPlan &plan) {
    const double us = flash_plan_us(rows, prefix, heads, head_dim, plan, &part_bytes);
    if (us < best_us && (plan.max_chunks == 1 || part_bytes <= workspace_bytes)) {
      best_us = us;
      best = plan;
    }
  };
  consider(FlashPlan{4, 0, 1});
  // Two and more rounds of the larger blocks: nothing idle to fill.
  if (workspace_bytes == 0 || ceil_div(rows, 8 * kQueriesPerWave) * heads >= 768)
    return best;
  const size_t tiles = (prefix + rows - 1) / kTileKeys + 1;
  for (uint32_t chunk : {8U, 12U, 16U, 24U, 32U, 48U, 64U, 96U, 128U, 192U, 256U, 384U, 768U,
                         1536U}) {
    const size_t chunks = (tiles + chunk - 1) / chunk;
    if (chunks < 2 || chunks > 64)
      continue;
    consider(FlashPlan{4, chunk, static_cast<uint32_t>(chunks)});
    consider(FlashPlan{8, chunk, static_cast<uint32_t>(chunks)});
  }
  return best;
}

template <int kD, typename O, int kWaves>
Status launch_flash_waves(const uint16_t *q, size_t q_plane, const uint16_t *k_cache,
                          const uint16_t *v_cache, size_t cache_plane, size_t capacity,
                          size_t rows, size_t prefix, size_t heads, const KeySplit &split, O out,
                          hipStream_t stream) {
  using Shape = FlashShape<kD, kWaves>;
  static_assert(Shape::kLdsBytes <= 64 * 1024, "default LDS limit, two blocks per CU");
  const size_t blocks = ceil_div(rows, Shape::kQueries) * heads * split.max_chunks;
  if (blocks > (1U << 31))
    return {ErrorCode::kInvalidArgument, "causal_attention: grid too large"};
  const auto kernel = capacity < (size_t{1} << 27)
                          ? flash_attention_kernel<kD, O, kWaves, false>
                          : flash_attention_kernel<kD, O, kWaves, true>;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(kWaves * 64),
                     Shape::kLdsBytes, stream, q, q_plane, k_cache, v_cache, cache_plane,
                     capacity, rows, prefix, heads, split, out);
  EVO_TRY(launch_status("flash_attention_kernel"));
  if (split.max_chunks == 1)
    return Status::Ok();
  hipLaunchKernelGGL((flash_combine_kernel<kD, O, kWaves>), dim3(ceil_div(rows * heads, 4)),
                     dim3(256), 0, stream, rows, prefix, heads, split, out);
  return launch_status("flash_combine_kernel");
}

template <int kD, typename O>
Status launch_flash(const uint16_t *q, size_t q_plane, const uint16_t *k_cache,
                    const uint16_t *v_cache, size_t cache_plane, size_t capacity, size_t rows,
                    size_t prefix, size_t heads, float *workspace, size_t workspace_bytes, O out,
                    hipStream_t stream) {
  // The parts are stored as float2.
  const bool usable = workspace != nullptr &&
                      reinterpret_cast<uintptr_t>(workspace) % sizeof(float2) == 0;
  const FlashPlan plan = plan_flash(rows, prefix, heads, kD, usable ? workspace_bytes : 0);
  const KeySplit split{plan.chunk_tiles, plan.max_chunks, workspace};
  if (plan.waves == 4)
    return launch_flash_waves<kD, O, 4>(q, q_plane, k_cache, v_cache, cache_plane, capacity, rows,
                                        prefix, heads, split, out, stream);
  return launch_flash_waves<kD, O, 8>(q, q_plane, k_cache, v_cache, cache_plane, capacity, rows,
                                      prefix, heads, split, out, stream);
}

// ---- Single-query (decode) attention, split over the keys: one block per
// (head, chunk of whole 64-key tiles). 16 lanes read a key's row of a plane
// (16 bytes each) and 8 lanes a V^T row's 64 positions, so every load of a
// tile, K and V, is a run of whole lines and all are in flight at once; the
// dots are F32, reduced over the lanes, the softmax runs on the tile's 64
// scores, and wave w sums the head's dimensions d % 32 / 8 == w (the V^T
// permutation swaps position bits 2 and 3, so column c holds key
// vt_column(c)). The chunk leaves (max, sum, o[d]); a second kernel per head
// rescales the chunks to the common max and sums them in chunk order.
// Full-softmax semantics as `src/cpu/model.cpp:510-544`.
// Bound by the latency of its loads at short prefixes (keys in chunks of 256,
// a key per lane, V after the softmax took 17.3 us at 1040 keys x 32 heads of
// 128, this 10.3) and by the cache's bytes at long ones (with the append, 32
// heads of 128: 8192 keys 175 -> 53.5 us, 32768 keys 772 -> 204, 131072 keys
// 2866 -> 802, 5.4 TB/s).
// Keys per chunk for which a workspace has to hold the parts; one that holds
// no more runs chunks of at least this length.
constexpr int kDecodeKeys = 256;
constexpr int kDecodeTile = 64;

template <int kD>
__global__ __launch_bounds__(256) void decode_attention_kernel(
    const uint16_t *__restrict__ q, size_t q_plane, const uint16_t *__restrict__ k_cache,
    const uint16_t *__restrict__ v_cache, size_t cache_plane, size_t capacity,
    size_t keys, size_t heads, int chunk_tiles, float *__restrict__ part) {
  constexpr int kRowLanes = kD / 8;                // lanes per key row
  constexpr int kKeysPerPass = 256 / kRowLanes;    // keys per block pass
  constexpr int kKPasses = kDecodeTile / kKeysPerPass > 0 ? kDecodeTile / kKeysPerPass : 1;
  constexpr int kVPasses = kD / 32;                // 32 dimensions per block pass
  __shared__ float score_s[kDecodeTile];
  __shared__ float p_s[kDecodeTile];
  const int tid = threadIdx.x, lane = tid & 63;
  const size_t chunk = blockIdx.x, h = blockIdx.y;
  const size_t width = heads * kD;
  const int row_lane = tid % kRowLanes, row_key = tid / kRowLanes;
  float qv[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    qv[e] = get_split(q, q + q_plane, h * kD + row_lane * 8 + e);
  const int v_lane = tid & 7, v_row = tid >> 3;
  float o[kVPasses] = {};
  float m = -INFINITY, l = 0.0F;
  const size_t tile0 = chunk * chunk_tiles;
  const size_t tile1 = min(tile0 + chunk_tiles, (keys + kDecodeTile - 1) / kDecodeTile);
  for (size_t t = tile0; t < tile1; ++t) {
    const size_t key0 = t * kDecodeTile;
    uint4 kh[kKPasses], kl[kKPasses], vh[kVPasses], vl[kVPasses];
#pragma unroll
    for (int i = 0; i < kKPasses; ++i) {
      const int key = i * kKeysPerPass + row_key;
      kh[i] = kl[i] = make_uint4(0, 0, 0, 0);
      if (key < kDecodeTile && key0 + key < keys) {
        const uint16_t *src = k_cache + (key0 + key) * width + h * kD + row_lane * 8;
        kh[i] = *reinterpret_cast<const uint4 *>(src);
        kl[i] = *reinterpret_cast<const uint4 *>(src + cache_plane);
      }
    }
#pragma unroll
    for (int i = 0; i < kVPasses; ++i) {
      const uint16_t *src = v_cache + (h * kD + i * 32 + v_row) * capacity + key0 + v_lane * 8;
      vh[i] = *reinterpret_cast<const uint4 *>(src);
      vl[i] = *reinterpret_cast<const uint4 *>(src + cache_plane);
    }
#pragma unroll
    for (int i = 0; i < kKPasses; ++i) {
      float kv[8], dot = 0.0F;
      split_floats(kh[i], kl[i], kv);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        dot = fmaf(qv[e], kv[e], dot);
#pragma unroll
      for (int offset = 1; offset < kRowLanes; offset <<= 1)
        dot += __shfl_xor(dot, offset, 64);
      const int key = i * kKeysPerPass + row_key;
      if (row_lane == 0 && key < kDecodeTile)
        score_s[key] = key0 + key < keys ? dot * (1.0F / sqrtf(static_cast<float>(kD)))
                                         : -INFINITY;
    }
    __syncthreads();
    // Every wave holds the tile's scores (lane = key): the same maximum and
    // sum in each.
    const float score = score_s[lane];
    float tile_max = score;
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1)
      tile_max = fmaxf(tile_max, __shfl_xor(tile_max, offset, 64));
    const float next = fmaxf(m, tile_max);
    const float reference = next == -INFINITY ? 0.0F : next;
    const float p = key0 + lane < keys ? expf(score - reference) : 0.0F;
    float sum = p;
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1)
      sum += __shfl_xor(sum, offset, 64);
    const float scale = t == tile0 ? 0.0F : expf(m - reference);
    l = t == tile0 ? sum : fmaf(l, scale, sum);
    m = next;
    if (tid < 64)
      p_s[lane] = p;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kVPasses; ++i) {
      float vv[8], acc = 0.0F;
      split_floats(vh[i], vl[i], vv);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        // Zero weights are skipped: columns of keys past the end may hold
        // unwritten cache.
        const float weight = p_s[vt_column(v_lane * 8 + e)];
        acc = weight != 0.0F ? fmaf(weight, vv[e], acc) : acc;
      }
      o[i] = t == tile0 ? acc : fmaf(o[i], scale, acc);
    }
  }
  float *dst = part + (h * gridDim.x + chunk) * (kD + 2);
#pragma unroll
  for (int i = 0; i < kVPasses; ++i) {
#pragma unroll
    for (int offset = 1; offset < 8; offset <<= 1)
      o[i] += __shfl_xor(o[i], offset, 64);
    if (v_lane == 0)
      dst[2 + i * 32 + v_row] = o[i];
  }
  if (tid == 0) {
    dst[0] = m;
    dst[1] = l;
  }
}

// 256 / kD groups of threads sum every group-th chunk, then each other.
template <int kD, typename O>
__global__ __launch_bounds__(256) void decode_combine_kernel(const float *__restrict__ part,
                                                             int chunks, O out) {
  constexpr int kGroups = 256 / kD;
  __shared__ float l_s[kGroups][kD], o_s[kGroups][kD], max_s[4];
  const size_t h = blockIdx.x;
  const int tid = threadIdx.x, d = tid % kD, group = tid / kD;
  const float *base = part + h * chunks * (kD + 2);
  float m = -INFINITY;
  for (int c = tid; c < chunks; c += 256)
    m = fmaxf(m, base[static_cast<size_t>(c) * (kD + 2)]);
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1)
    m = fmaxf(m, __shfl_xor(m, offset, 64));
  if ((tid & 63) == 0)
    max_s[tid >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(max_s[0], max_s[1]), fmaxf(max_s[2], max_s[3]));
  const float reference = m == -INFINITY ? 0.0F : m;
  float l = 0.0F, o = 0.0F;
#pragma unroll 4
  for (int c = group; c < chunks; c += kGroups) {
    const float *src = base + static_cast<size_t>(c) * (kD + 2);
    const float scale = expf(src[0] - reference);
    l = fmaf(src[1], scale, l);
    o = fmaf(src[2 + d], scale, o);
  }
  l_s[group][d] = l;
  o_s[group][d] = o;
  __syncthreads();
  if (group != 0)
    return;
#pragma unroll
  for (int g = 1; g < kGroups; ++g) {
    l += l_s[g][d];
    o += o_s[g][d];
  }
  put(out, h * kD + d, o / l);
}

template <int kD, typename O>
Status launch_decode(const uint16_t *q, size_t q_plane, const uint16_t *k_cache,
                     const uint16_t *v_cache, size_t cache_plane, size_t capacity, size_t keys,
                     size_t heads, float *workspace, size_t workspace_bytes, O out,
                     hipStream_t stream) {
  // One tile per chunk below 4096 blocks (16 per CU), then the most tiles that
  // leave 2048; no more than 512 chunks to combine, and parts that fit.
  const size_t tiles = ceil_div(keys, kDecodeTile);
  const size_t part = heads * (kD + 2) * sizeof(float);
  size_t chunk_tiles = std::max<size_t>(1, tiles * heads / 2048);
  chunk_tiles = std::max<size_t>(chunk_tiles, ceil_div(tiles, 512));
  if ((tiles + chunk_tiles - 1) / chunk_tiles * part > workspace_bytes)
    chunk_tiles = std::max<size_t>(chunk_tiles, kDecodeKeys / kDecodeTile);
  const unsigned chunks = static_cast<unsigned>((tiles + chunk_tiles - 1) / chunk_tiles);
  hipLaunchKernelGGL(decode_attention_kernel<kD>, dim3(chunks, heads), dim3(256), 0, stream, q,
                     q_plane, k_cache, v_cache, cache_plane, capacity, keys, heads,
                     static_cast<int>(chunk_tiles), workspace);
  EVO_TRY(launch_status("decode_attention_kernel"));
  hipLaunchKernelGGL((decode_combine_kernel<kD, O>), dim3(heads), dim3(256), 0, stream,
                     workspace, static_cast<int>(chunks), out);
  return launch_status("decode_combine_kernel");
}

template <typename O>
Status launch_attention(const uint16_t *q, size_t q_plane, const uint16_t *k_cache,
                        const uint16_t *v_cache, size_t cache_plane, size_t capacity,
                        size_t rows, size_t prefix, size_t heads, size_t head_dim,
                        float *workspace, size_t workspace_bytes, O out, hipStream_t stream) {
  switch (head_dim) {
  case 16:
    hipLaunchKernelGGL((attention_kernel<16, O>), dim3(ceil_div(rows, 64), heads), dim3(256),
                       0, stream, q, q_plane, k_cache, v_cache, cache_plane, capacity, rows,
                       prefix, heads, out);
    return launch_status("attention_kernel");
  case 32:
    return launch_flash<32, O>(q, q_plane, k_cache, v_cache, cache_plane, capacity, rows,
                               prefix, heads, workspace, workspace_bytes, out, stream);
  case 64:
    return launch_flash<64, O>(q, q_plane, k_cache, v_cache, cache_plane, capacity, rows,
                               prefix, heads, workspace, workspace_bytes, out, stream);
  case 128:
    return launch_flash<128, O>(q, q_plane, k_cache, v_cache, cache_plane, capacity, rows,
                               prefix, heads, workspace, workspace_bytes, out, stream);
  default:
    return {ErrorCode::kUnsupported,
            "causal_attention: head_dim must be 16, 32, 64 or 128"};
  }
}

}  // namespace

Status qkv_rope(const float *projected, size_t rows, size_t width, size_t heads,
                bool column_split, const float *inv_freq, float rope_scale,
                size_t prefix, uint16_t *q, size_t q_plane, uint16_t *k_cache,
                uint16_t *v_cache, size_t cache_plane, size_t capacity, hipStream_t stream,
                int *v_range_flag) {
  if (projected == nullptr || inv_freq == nullptr || q == nullptr ||
      k_cache == nullptr || v_cache == nullptr || rows == 0 || heads == 0 ||
      width % heads != 0 || (width / heads) % 2 != 0 || !(rope_scale > 0.0F) ||
      q_plane < rows * width || capacity % kKeys != 0 || prefix + rows > capacity ||
      cache_plane < capacity * width)
    return {ErrorCode::kInvalidArgument, "qkv_rope: invalid arguments"};
  const size_t half = width / heads / 2;
  if (256 % half != 0 || rows > (1U << 31))
    return {ErrorCode::kInvalidArgument, "qkv_rope: head_dim / 2 must divide 256"};
  const size_t value_blocks = static_cast<size_t>(ceil_div(rows, 64)) * ceil_div(width, 64);
  // Four pairs or channels per thread where every run starts on 16 bytes of
  // the projection and 8 of a plane.
  const bool vec = half % 4 == 0 && reinterpret_cast<uintptr_t>(projected) % 16 == 0 &&
                   (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_cache)) % 8 ==
                       0 &&
                   q_plane % 4 == 0 && cache_plane % 4 == 0;
  // A few rows: a block per group of heads instead of one per row.
  const size_t head_step = 256 / (half / (vec ? 4 : 1));
  const size_t row_parts = rows >= 256 ? 1 : ceil_div(heads, head_step);
  const size_t blocks = value_blocks + rows * row_parts;
  if (blocks > (1U << 31))
    return {ErrorCode::kInvalidArgument, "qkv_rope: grid too large"};
  const QkvAppend append{projected, rows, width, heads, static_cast<int>(half),
                         column_split ? 1 : 0, inv_freq, rope_scale, prefix, q, q_plane,
                         k_cache, v_cache, cache_plane, capacity, v_range_flag,
                         static_cast<unsigned>(value_blocks), static_cast<unsigned>(row_parts)};
  hipLaunchKernelGGL(vec ? append_qkv_kernel<4> : append_qkv_kernel<1>,
                     dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, append);
  return launch_status("append_qkv_kernel");
}

Status causal_attention(const uint16_t *q, size_t q_plane, const uint16_t *k_cache,
                        const uint16_t *v_cache, size_t cache_plane, size_t capacity,
                        size_t rows, size_t prefix, size_t heads, size_t head_dim,
                        float *out_f32, uint16_t *out_hi, uint16_t *out_lo,
                        hipStream_t stream, float *workspace, size_t workspace_bytes,
                        bool out_f16) {
  if (q == nullptr || k_cache == nullptr || v_cache == nullptr ||
      (out_f32 == nullptr && out_hi == nullptr) || rows == 0 || heads == 0 ||
      heads > 65535 || q_plane < rows * heads * head_dim || capacity % kKeys != 0 ||
      prefix + rows > capacity || cache_plane < capacity * heads * head_dim)
    return {ErrorCode::kInvalidArgument, "causal_attention: invalid arguments"};
  // One query with a workspace for the chunk partials: split over the keys.
  const size_t keys = prefix + 1;
  if (rows == 1 && workspace != nullptr &&
      (head_dim == 32 || head_dim == 64 || head_dim == 128) &&
      heads * ceil_div(keys, kDecodeKeys) * (head_dim + 2) * sizeof(float) <= workspace_bytes) {
    auto run = [&](auto out) -> Status {
      switch (head_dim) {
      case 32:
        return launch_decode<32>(q, q_plane, k_cache, v_cache, cache_plane, capacity, keys,
                                 heads, workspace, workspace_bytes, out, stream);
      case 64:
        return launch_decode<64>(q, q_plane, k_cache, v_cache, cache_plane, capacity, keys,
                                 heads, workspace, workspace_bytes, out, stream);
      default:
        return launch_decode<128>(q, q_plane, k_cache, v_cache, cache_plane, capacity, keys,
                                  heads, workspace, workspace_bytes, out, stream);
      }
    };
    if (out_f32 != nullptr)
      return run(out_f32);
    if (out_f16)
      return run(F16Plane{out_hi});
    return run(SplitOut{out_hi, out_lo});
  }
  if (out_f32 != nullptr)
    return launch_attention(q, q_plane, k_cache, v_cache, cache_plane, capacity, rows, prefix,
                            heads, head_dim, workspace, workspace_bytes, out_f32, stream);
  if (out_f16)
    return launch_attention(q, q_plane, k_cache, v_cache, cache_plane, capacity, rows, prefix,
                            heads, head_dim, workspace, workspace_bytes, F16Plane{out_hi}, stream);
  return launch_attention(q, q_plane, k_cache, v_cache, cache_plane, capacity, rows, prefix, heads,
                          head_dim, workspace, workspace_bytes, SplitOut{out_hi, out_lo}, stream);
}

}  // namespace evo::hip
