// SPDX-License-Identifier: Apache-2.0
// The rules by which launches choose their shape, as functions of the sizes
// (host code; the reasons and measurements stand at the definitions). The
// dispatches call them, and so do the tests, through testing.cpp.
#pragma once

#include <cstddef>

namespace evo::hip {

// Rows per segment of the HCS row stream (hyena.hip).
unsigned hcs_stream_segment(size_t width, size_t length, bool f32_exact);

}  // namespace evo::hip
