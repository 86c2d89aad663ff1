// Positions of a row's entries for a group of lanes that walks them in steps
// past the row's end.  A matrix holds up to 2^31 - 1 entries, so a position past
// the end of one of its last rows does not fit 32 bits with a sign: the walks
// count from the row's first entry, unsigned.  (constexpr: device and host.)
#pragma once

#include <cstdint>

namespace gpdev {

// Entries of the row [b, e).
constexpr uint32_t row_length(int32_t b, int32_t e) { return static_cast<uint32_t>(e) - static_cast<uint32_t>(b); }

// Entry o of the row [b, e), the last one where o is past it (e > b).
constexpr int32_t row_entry(int32_t b, int32_t e, uint32_t o) {
  const uint32_t n = row_length(b, e);
  return b + static_cast<int32_t>(o < n ? o : n - 1);
}

}  // namespace gpdev
