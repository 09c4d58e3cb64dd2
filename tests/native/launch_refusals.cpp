// Launches that no kernel is built for: the launchers (the built kernels' object) refuse them before the runtime is asked for anything.
#include "kernels.h"

#include <cstdio>

using namespace tbamd;

static int gFailures = 0;

int main() {
  // Rank tiles keep all leaves in LDS: the walk that looks them up outside is not built for them, the plain one would read other
  // bytes in their place.
  for (int tileMode : {2, 3}) // (one-byte and two-byte ranks)
    for (int interleave : {1, 2, 4, 8})
      for (int splitBlocks : {0, 2})
        for (int classes : {0, 4})
          for (int own : {0, 1})
            for (bool direct : {false, true}) {
              if (own && !classes) continue;
              double partial = 0.0;
              float out = 0.0f;
              WalkParams p;
              p.s.rows = 200;
              p.s.rowsPerBlock = 64;
              p.s.treeThreads = 16;
              p.s.numFeatures = 20;
              p.s.numGroups = 2;
              p.s.groupRegionBytes = 16384;
              p.s.numClasses = classes;
              p.s.ownClasses = own;
              p.s.leavesOutside = 1;
              p.directStaging = direct;
              p.splitBlocks = splitBlocks;
              p.partial = &partial;
              p.out = &out;
              const hipError_t e = LaunchWalkRowsLds(p, interleave, tileMode, 64 * 1024, nullptr);
              if (e == hipErrorInvalidValue) continue;
              ++gFailures;
              std::printf("tile mode %d, %d trees a lane, %d split blocks, %d classes, own %d, direct %d: %s\n", tileMode, interleave, splitBlocks, classes, own,
                          direct, hipGetErrorName(e));
            }
  if (gFailures) return 1;
  std::printf("ok\n");
  return 0;
}
