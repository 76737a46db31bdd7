// kmst_walks.hpp -- bounds of the direct solve's walks to a root.
#pragma once

#include <cstdint>

namespace kmst {

// Rounds of a solve at most: every round at least halves the components that
// have edges, so more is a corrupted forest.
constexpr std::uint32_t UNION_ROUNDS_MAX = 200;

// Weights in order along a path hook it into one chain, which walks of the list's
// entries may not shorten for each other.  A walk longer than this stops, and
// shorten_chains takes all vertices to their roots before the round goes on.  A
// step takes some 0.9 us, the passes 15 us up to 10^5 vertices and a time that
// grows with n past that, hence the limit.  10^6 vertices, descending weights along a path,
// heavier chords: 0.44 ms, 116 where the round loop took over after 1024 steps
// (114 alone); 9000 vertices of a band 160 us, 1265 (205); a grid of 300 x 300
// 166 us, 313 with walks alone (250).  Random weights stay below
// (of 162 graphs of 8200 to 200000 vertices one met a limit of 8, none one of 10).
constexpr std::uint32_t WALK_DEEP_MIN = 10;
constexpr int WALK_DEEP_SHIFT = 15;
constexpr std::uint32_t walk_deep(std::uint32_t n) {
  return WALK_DEEP_MIN + (n >> WALK_DEEP_SHIFT);
}

// Steps of a walk in a whole forest: after a round every vertex that hooked in it is
// within walk_deep of a root, and a later round adds as much.  The symmetry sums
// can collide, and hooks of records that are not symmetric may close a cycle, which
// rounds on dense ids do not meet: a walk past this is one, and the solve ends with an error.
// With a bound of 2^26 steps each such walk took a minute.
constexpr std::uint32_t walk_limit(std::uint32_t n) {
  return UNION_ROUNDS_MAX * (walk_deep(n) + 2);
}

}  // namespace kmst
