// SPDX-License-Identifier: Apache-2.0
// The rules by which launches choose their shape, as functions of the sizes
// (host code; the reasons and measurements stand at the definitions). The
// dispatches call them, and so do the tests, through testing.cpp.
#pragma once

#include <cstddef>

namespace evo::hip {

// Rows per segment of the HCS row stream (hyena.hip).
unsigned hcs_stream_segment(size_t width, size_t length, bool f32_exact);

// Whether the HCM row stream takes filter groups that are no multiple of 16
// (hyena.hip), rows and outputs aligned.
bool hcm_stream_two_groups(size_t group_size, size_t length, int taps, bool f32);

}  // namespace evo::hip
