// CPU check of the forwards' workgroup-to-row mapping (launch_plan.h: xcd_item, xcd_run_log2), built
// by tests/test_xcd_runs.py: a permutation of the blocks for every grid size, whose whole spans
// give each XCD (block index mod 8) a run of consecutive items.
#include <stdio.h>
#include <stdlib.h>

#include <vector>

#include "launch_plan.h"

int main() {
  using namespace vg_plan;
  const uint32_t sizes[] = {1, 7, 8, 9, 63, 64, 127, 128, 129, 511, 512, 513, 4097, 16384, 70001};
  for (uint32_t n : sizes) {
    for (int run = 0; run <= kXcdRunMaxLog2; ++run) {
      std::vector<char> seen(n, 0);
      for (uint32_t b = 0; b < n; ++b) {
        const uint32_t i = xcd_item(b, n, run);
        if (i >= n || seen[i]) return printf("n=%u run=%d b=%u item=%u\n", n, run, b, i), 1;
        seen[i] = 1;
        const uint32_t span = 8u << run;
        if (b / span < n / span && (i % span) >> run != b % 8)
          return printf("run of another XCD: n=%u run=%d b=%u item=%u\n", n, run, b, i), 1;
        if (b / span >= n / span && i != b) return printf("tail moved: n=%u b=%u\n", n, b), 1;
      }
    }
  }
  // runs near 256 KiB of a stream, and never past the largest
  for (int64_t bytes = 1; bytes <= (1 << 20); bytes = bytes * 3 / 2 + 1) {
    for (int groups = 1; groups <= 4; ++groups) {
      const int run = xcd_run_log2(bytes, groups);
      const int64_t moved = (bytes * groups) << run;
      if (run < 0 || run > kXcdRunMaxLog2 || (run > 0 && moved * 3 > kXcdRunBytes * 4) ||
          (run < kXcdRunMaxLog2 && moved * 3 <= kXcdRunBytes * 2))
        return printf("run_log2(%lld, %d) = %d\n", (long long)bytes, groups, run), 1;
    }
  }
  if (xcd_run_log2(8192, 1) != 5) return printf("8 KiB rows\n"), 1;
  // wide rows of the generic kernel keep their block's index, narrower ones go in runs
  if (xcd_run_log2(22010, 1, true) != 0 || xcd_run_log2(65536, 1, true) != 0 ||
      xcd_run_log2(18002, 1, true) != xcd_run_log2(18002, 1))
    return printf("generic rows\n"), 1;
  printf("xcd_run_check ok\n");
  return 0;
}
