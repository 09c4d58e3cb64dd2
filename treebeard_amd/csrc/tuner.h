// Launch-parameter tuner: picks the kernel and its shape from the model's
// statistics and the batch size.  It stands where the reference has its
// scheduling language and GPU auto-tuner (src/schedule/schedule.h,
// src/mlir/GPUAutoSchedule.cpp:597-624 heuristic subset, :799-934 timed search).
#pragma once

#include "forest.h"
#include "options.h"
#include "packer.h"

#include <vector>

namespace tbamd {

struct DeviceLimits {
  int32_t computeUnits = 256;
  int32_t ldsBytesPerBlock = 160 * 1024;
};

// What the compiler options ask of the walk itself (CompilerOptions::tileSize, tilingType and the peeled
// code generation switch); copied into the plan.
struct WalkOptions {
  int32_t tileSize = 1;
  int32_t tiling = 0;     // 0 uniform, 1 probabilistic, 2 hybrid
  bool peelWalks = false;
};

// What a row-parallel walk over `rowBlocks` row blocks takes on the device, in microseconds: enough to choose between
// launch shapes of one plan, not to predict a time.  Fitted to MI355X timings of 100 to 1000 trees on 10 to 90 features
// and 2048 to 200000 rows: a lock-step level of 64 rows occupies a compute unit's LDS for 5.4 cycles, shared by the
// blocks on it; a tree group costs 1.35 us of copy and barriers that a second block hides but for 0.9; partial sums
// cost a finalize launch of 5 us.
struct WalkShape {
  int64_t rowBlocks = 1;
  int32_t rowsPerBlock = 256, numFeatures = 1;
  double levels = 0.0;        // lock-step levels of one row over the whole forest
  double groups = 1.0;        // tree groups of the whole forest
  int32_t computeUnits = 256;
  int32_t blocksPerUnit = 2;  // that run at once
};
double SlicedWalkMicros(const WalkShape &shape, int32_t treeSlices); // a block per row block and tree slice
double SplitWalkMicros(const WalkShape &shape);                      // row blocks x groups split evenly over the blocks that run at once

// Analytic choice; `overrides` (may be null) pins what the caller set.  Tile sizes above 1 always get the
// row-parallel kernel on f32 rows (the only one that walks tiles) and fail when its row tile does not fit.
LaunchPlan ChoosePlan(const Forest &forest, int64_t batchSize, const GPUAutoScheduleOptions *overrides,
                      const DeviceLimits &limits, const WalkOptions &walk = WalkOptions());

// Whether `plan` can defer the tails of its walks (LaunchPlan::deferTails: the scalar row-parallel kernel on an f32
// tile with byte offsets, a model without classes); when it can, the plan's tree groups give up the LDS the stub
// feature's column and the waves' queues take.  The caller sets the flag.
bool DeferTailsFit(const Forest &forest, LaunchPlan *plan);
// The block shape of forests of a few KB (ChoosePlan), which has no deferred tails.
bool SmallForestBlocks(const Forest &forest, const LaunchPlan &plan);

// A forest with a tree too big for an LDS tree group (LaunchPlan::Kernel::kGlobalWalk), walked with deferred tails instead of
// node by node from global memory: the tops of its trees fit.  Sets a plan for PackWithCuts and the level every tree is cut
// at; false where the form cannot hold the forest (classes, rows too wide, too many nodes below the cuts).
bool ChooseDeepWalk(const Forest &forest, const DeviceLimits &limits, LaunchPlan *plan, std::vector<int32_t> *cuts);
// How many blocks share a row block's tree groups.
int32_t DeepWalkSlices(int64_t rowBlocks, int64_t groups, const DeviceLimits &limits);

// A plan of one group size out of a file: where its classes are the tree threads' own and it counts on the meeting place that they
// leave, that size becomes LaunchPlan::ownGroupBytes and groupBytes the one beside the place.  The packed groups stay the same.
void SeparateGroupSizes(const Forest &forest, const HitCountProfile *profile, const DeviceLimits &limits, LaunchPlan *plan);

// Candidate plans for the timed search (the analytic choice comes first).
std::vector<LaunchPlan> CandidatePlans(const Forest &forest, int64_t batchSize, const DeviceLimits &limits,
                                       const WalkOptions &walk = WalkOptions());

} // namespace tbamd
