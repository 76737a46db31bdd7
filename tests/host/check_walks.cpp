// Bounds of the direct solve's walks: a forest of hooks never meets them, and
// a walk round a cycle ends before the other workgroups' waits do (10 s).
#include <cstdio>
#include <initializer_list>

#include "kmst_walks.hpp"

int main() {
  int bad = 0;
  for (int b = 1; b <= 28; ++b)
    for (std::uint32_t n : {(1u << b) - 1, 1u << b}) {
      std::uint64_t depth = 0;  // the deepest vertex
      for (std::uint64_t roots = n; roots > 1; roots /= 2)
        depth += kmst::walk_deep(n) + 2;  // a walk's last steps find the root and stay there
      if (depth > kmst::walk_limit(n)) {
        std::printf("n %u: a walk of %llu steps is refused\n", n, (unsigned long long)depth);
        ++bad;
      }
      const double seconds = 1e-6 * kmst::walk_limit(n);
      if (seconds > 5) {
        std::printf("n %u: a cycle is walked for %.1f s\n", n, seconds);
        ++bad;
      }
    }
  if (!bad) std::printf("ok (walks)\n");
  return bad != 0;
}
