// SPDX-License-Identifier: Apache-2.0
// C entry points for this repository's tests, in a library of their own
// (lib/libevo_hip_testing.so): the launch rules as functions of the sizes.
// No part of the product's interface.
#include "launch_rules.hpp"

#define EVO_TEST_API extern "C" __attribute__((visibility("default")))

EVO_TEST_API unsigned evo_test_hcs_stream_segment(size_t width, size_t length, int f32_exact) {
  return evo::hip::hcs_stream_segment(width, length, f32_exact != 0);
}

EVO_TEST_API int evo_test_hcm_stream_two_groups(size_t group_size, size_t length, int taps,
                                                int f32) {
  return evo::hip::hcm_stream_two_groups(group_size, length, taps, f32 != 0) ? 1 : 0;
}
