// The placement rule (xcd_run, mprgp_host.h) over every launch size and tile
// shape: prints the first violation and returns 1.
#include <cstdio>

#include "../../mprgp_amd/csrc/mprgp_host.h"

using namespace mprgp;

int main() {
  for (int span = 1; span <= 16; span *= 2)
    for (int n = 1; n <= 5000; ++n) {
      int grid = 64;
      while (grid < n || (grid < 256 && grid < 8 * n)) grid *= 2;
      const int run = xcd_run(n, grid, span);
      const bool pow2 = run > 0 && (run & (run - 1)) == 0;
      // what an XCD has side by side: 32 slices, or the 4 tiles of the smallest run
      const bool few = run <= 4 || run * span <= 32;
      const bool fits = run * 8 <= grid;
      const bool shared = n > 1024 ? run == 4 : true;
      if (!pow2 || !few || !fits || !shared) {
        std::printf("%d tiles of %d slices, %d slots: runs of %d\n", n, span, grid, run);
        return 1;
      }
      if (span == 1 && n <= 256 && run != (grid / 8 < 32 ? grid / 8 : 32)) {
        std::printf("%d tiles of one slice: runs of %d\n", n, run);
        return 1;
      }
    }
  return 0;
}
