// Index expressions that 32-bit arithmetic does not hold, usable on the host.
#pragma once
#include <cstdint>

namespace p3d {

// First entry of row `row` of a coordinate table [N, 3].  N < 2^31, so the row
// fits in 32 bits; three times the row does not from 715,827,883 rows on.
constexpr int64_t coord_start(int64_t row) { return 3 * row; }

}  // namespace p3d
