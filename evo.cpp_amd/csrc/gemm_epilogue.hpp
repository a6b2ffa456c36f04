// SPDX-License-Identifier: Apache-2.0
// Epilogue description shared by the dense-linear kernels (device code;
// included by the .hip sources).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "ops.hpp"

namespace evo::hip {

struct Epilogue {
  int mode;              // GemmEpilogue
  const uint16_t *bias;  // BF16 [N]
  const float *residual; // F32 [M, ldc]
  int gelu;              // gated: erf-GELU on the l1 half
  int gated_width;       // gated: valid output columns
};

__device__ inline float gelu_erf(const float x) {
  return 0.5F * x * (1.0F + erff(x * 0.7071067811865475244F));
}

}  // namespace evo::hip
