// The host-side arithmetic of kernels.h that the launchers and the runner share, over its whole range.
#include "kernels.h"

#include <cstdio>

using namespace tbamd;

static int gFailures = 0;
#define EXPECT(cond, ...)                                                                                              \
  do {                                                                                                                 \
    if (!(cond) && ++gFailures < 20) std::printf("FAILED %s: ", #cond), std::printf(__VA_ARGS__), std::printf("\n"); \
  } while (0)

// Every forest: the batches up to its limit fit a block's LDS and its lanes (a lane per row finishes the classes), and no
// wave adds more sums than 0.4 us each are worth.
static void FewRows() {
  for (int classes : {0, 2, 3, 6, 12, 40, 128})
    for (int trees = 1; trees <= 1200; trees += trees < 40 ? 1 : 97)
      for (int features : {1, 4, 28, 600, 2047, 20000})
        for (int depth : {0, 1, 3, 6, 8, 14, 30}) {
          const int64_t limit = FewRowsLimit(features, trees, classes, depth);
          EXPECT(limit >= 0 && limit <= kFewRowsWork, "%d classes %d trees %d features depth %d", classes, trees, features, depth);
          for (int64_t rows : {(int64_t)1, limit / 3, limit - 1, limit}) {
            if (rows < 1 || rows > limit) continue;
            const FewRowsShape s = ShapeOfFewRows(rows, features, trees, classes);
            const int64_t sums = (int64_t)s.rowsPerBlock * (classes ? classes : 1);
            EXPECT(s.threads % 64 == 0 && s.threads <= 1024 && s.ldsBytes <= kFewRowsLds, "%d classes %d trees %d features depth %d: %lld rows",
                   classes, trees, features, depth, (long long)rows);
            EXPECT(s.rowsPerBlock <= s.threads, "%d classes %d trees %d features depth %d: %lld rows, %d a block of %d lanes", classes, trees, features,
                   depth, (long long)rows, s.rowsPerBlock, s.threads);
            EXPECT(rows < limit || (sums - 1) / (s.threads / 64) * 0.4 <= 6.5 + 1.1 * classes, "%d classes %d trees %d features depth %d: %lld rows", classes,
                   trees, features, depth, (long long)rows);
          }
        }
}

int main() {
  FewRows();
  if (gFailures) return 1;
  std::printf("ok\n");
  return 0;
}
