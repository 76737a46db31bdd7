// kmst_rows.hpp -- rows of the input: a vertex's first position, its end << 32.
#pragma once

#include <cstdint>

namespace kmst {

// Bounds of a search for the place of an id in a row: [first, last], both
// positions of the input also where the row is empty (0, 0).  The symmetry sums
// can collide, so a record may point at a vertex that has no records.
constexpr std::uint32_t row_first(std::uint64_t span) { return static_cast<std::uint32_t>(span); }
constexpr std::uint32_t row_last(std::uint64_t span) {
  const std::uint32_t end = static_cast<std::uint32_t>(span >> 32);
  return end ? end - 1 : 0;
}

}  // namespace kmst
