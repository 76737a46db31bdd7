// Bounds of the direct solve's walks: a forest of hooks never meets them, and
// a walk round a cycle ends before the other workgroups' waits do (10 s).
#include <cstdio>

#include "kmst_walks.hpp"

int main() {
  int bad = 0;
  for (int b = 1; b <= 28; ++b) {
    std::uint64_t depth = 0;  // the deepest vertex
    for (std::uint64_t roots = std::uint64_t{1} << b; roots > 1; roots /= 2)
      depth += kmst::WALK_DEEP + 2;  // a walk's last steps find the root and stay there
    if (depth > kmst::WALK_LIMIT) {
      std::printf("2^%d vertices: a walk of %llu steps is refused\n", b, (unsigned long long)depth);
      ++bad;
    }
  }
  const double seconds = 1e-6 * kmst::WALK_LIMIT;
  if (seconds > 5) {
    std::printf("a cycle is walked for %.1f s\n", seconds);
    ++bad;
  }
  if (!bad) std::printf("ok (walks)\n");
  return bad != 0;
}
