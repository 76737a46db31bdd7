// kmst_walks.hpp -- bounds of the direct solve's walks to a root.
#pragma once

#include <cstdint>

namespace kmst {

// Rounds of a solve at most: every round at least halves the components that
// have edges, so more is a corrupted forest.
constexpr std::uint32_t UNION_ROUNDS_MAX = 200;

// Weights in order along a path hook it into one chain, which walks of the list's
// entries may not shorten for each other.  A walk longer than this stops, and
// shorten_chains takes all vertices to their roots before the round goes on.  Both cost
// with n: at 10^6 vertices a step of all walks takes 4 to 11 us, the passes 15 to 30; hence
// one limit for all sizes.  Bands 8 wide, the vertices in random order, with limits of
// 10, 12, 16 and 42: 1301, 1328, 1415 and 1778 us at 2^20 vertices; at 2^22 2705, 2756,
// 2900 and (with 138) 4191.  Random weights stay below: of 76 random, geometric and
// hyperbolic graphs of 2^17 to 2^24 vertices two met a limit of 10 (1 % slower), none one of 14.
constexpr std::uint32_t WALK_DEEP = 12;

// Steps of a walk in a whole forest: after a round every vertex that hooked in it is
// within WALK_DEEP of a root, and a later round adds as much.  The symmetry sums
// can collide, and hooks of records that are not symmetric may close a cycle, which
// rounds on dense ids do not meet: a walk past this is one, and the solve ends with an error.
// With a bound of 2^26 steps each such walk took a minute.
constexpr std::uint32_t WALK_LIMIT = UNION_ROUNDS_MAX * (WALK_DEEP + 2);

}  // namespace kmst
