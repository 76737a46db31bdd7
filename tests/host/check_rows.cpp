// The search for a forward record's position in a row, as the direct solve
// makes it, reads the input at its positions only, in an empty row too.
#include <cstdio>
#include <vector>

#include "kmst_rows.hpp"

int main() {
  const std::vector<std::uint32_t> dst{2, 5, 9, 0, 7};  // rows [0, 3), [3, 5), then none
  const std::uint64_t rows[] = {std::uint64_t{3} << 32, std::uint64_t{5} << 32 | 3, 0};
  int bad = 0;
  for (std::uint64_t span : rows)
    for (std::uint32_t id : {0u, 2u, 5u, 7u, 9u, 10u, 0xFFFFFFFEu}) {
      std::uint32_t lo = kmst::row_first(span), hi = kmst::row_last(span);
      while (lo < hi) {
        const std::uint32_t mid = lo + (hi - lo) / 2;
        if (mid >= dst.size()) {
          std::printf("row %llx, id %u: reads position %u\n", (unsigned long long)span, id, mid);
          return 1;
        }
        if (dst[mid] < id) lo = mid + 1;
        else hi = mid;
      }
      bad += lo >= dst.size();
      const std::uint32_t end = static_cast<std::uint32_t>(span >> 32);
      for (std::uint32_t i = static_cast<std::uint32_t>(span); i < end; ++i)
        if (dst[i] == id) bad += lo != i;  // what is there is found
    }
  if (!bad) std::printf("ok (rows)\n");
  return bad != 0;
}
