#include "tuner.h"

#include <algorithm>
#include <cmath>

namespace tbamd {

namespace {

int32_t FloorPow2(int64_t v) {
  int32_t p = 1;
  while ((int64_t)p * 2 <= v) p *= 2;
  return p;
}

// Largest rows-per-block (power of two, >= 64) whose transposed row tile keeps
// 16-bit feature offsets and leaves room for a tree group.
bool RowTileFits(int32_t numFeatures, int32_t rowsPerBlock, int32_t ldsBytes, bool *offsetsInWords) {
  const int64_t words = (int64_t)(numFeatures + 1) * rowsPerBlock;
  if (words > 0xFFFF) return false;
  if (words * 4 + 16 * 1024 > ldsBytes) return false; // keep at least 16 KB for trees
  *offsetsInWords = words * 4 > 0xFFFF;
  return true;
}


// A block that takes `share` of the forest through its rows, with `together` blocks on its compute unit.
double BlockMicros(const WalkShape &w, double share, int together) {
  const double rowBytes = (double)w.rowsPerBlock * w.numFeatures * 4;
  const double stage = 2.0 + (together > 1 ? rowBytes * together * w.computeUnits / 4e6 : rowBytes / 20e3);
  const double walk = w.levels * (w.rowsPerBlock / 64.0) * 5.4 / 2400.0;
  return stage + share * (together * walk + w.groups * (together > 1 ? 0.9 : 1.35));
}
constexpr double kFinalizeMicros = 5.0;

int64_t BiggestTreeNodes(const Forest &forest) {
  int64_t biggest = 0;
  for (auto &t : forest.trees) biggest = std::max<int64_t>(biggest, (int64_t)t.NumNodes());
  return biggest;
}

// Rows row-major in LDS, several lanes per row.
LaunchPlan ChooseTreeParallelPlan(const Forest &forest, int64_t batchSize, const GPUAutoScheduleOptions *ov,
                                  const DeviceLimits &limits) {
  LaunchPlan plan;
  plan.kernel = LaunchPlan::Kernel::kTreeParallel;
  plan.interleave = 1;
  if (ov && ov->treeWalkInterleaveFactor > 0)
    plan.interleave = std::min(kMaxInterleave, FloorPow2(ov->treeWalkInterleaveFactor));
  const int64_t rowBytes = (int64_t)(forest.numFeatures + 1) * 4;
  const int64_t need = (BiggestTreeNodes(forest) + 2) * kNodeBytes;
  if (need > 65536) throw Error("a tree does not fit one LDS tree group");
  int64_t group = std::max<int64_t>(need, 24 * 1024);
  const int64_t reserve = 4096; // reduction scratch and class sums
  if (rowBytes + group + reserve > limits.ldsBytesPerBlock) group = need;
  if (rowBytes + group + reserve > limits.ldsBytesPerBlock)
    throw Error("a row of " + std::to_string(forest.numFeatures) + " features does not fit LDS next to a tree group");
  int64_t rows = FloorPow2((limits.ldsBytesPerBlock - group - reserve) / rowBytes);
  rows = std::min<int64_t>(rows, 16);
  if (ov && ov->numRowsPerTB > 0) rows = std::min<int64_t>(rows, FloorPow2(ov->numRowsPerTB));
  if (batchSize > 0) rows = std::min<int64_t>(rows, FloorPow2(std::max<int64_t>(batchSize, 1) * 2 - 1));
  plan.rowsPerBlock = (int32_t)std::max<int64_t>(rows, 1);
  plan.treeLanes = std::max(1, 256 / plan.rowsPerBlock);
  // narrow rows leave LDS for bigger groups
  const int64_t rowTile = rowBytes * plan.rowsPerBlock;
  group = std::max<int64_t>(group, std::min<int64_t>(65536, (limits.ldsBytesPerBlock / 2 - rowTile - reserve)));
  group = std::min<int64_t>(group, 256LL * plan.ThreadsPerBlock()); // 16 prefetch registers of 16 bytes per lane
  if (group < need) throw Error("the biggest tree does not fit the group prefetch registers of this block shape");
  plan.groupBytes = (int32_t)(std::min<int64_t>(group, 65536) & ~15);

  const int64_t rowBlocks = std::max<int64_t>(1, (batchSize + plan.rowsPerBlock - 1) / plan.rowsPerBlock);
  const int64_t totalBytes = (int64_t)forest.NumNodes() * kNodeBytes;
  int64_t groups = std::max<int64_t>(1, (totalBytes + plan.groupBytes - 1) / plan.groupBytes);
  int64_t slices = 1;
  const int64_t wantBlocks = 2LL * limits.computeUnits;
  if (rowBlocks < wantBlocks) slices = (wantBlocks + rowBlocks - 1) / rowBlocks;
  if (ov && ov->numTreeThreads > 0) slices = ov->numTreeThreads;
  slices = std::min<int64_t>(slices, std::max<int64_t>(1, totalBytes / 8192)); // at least 8 KB of trees per slice
  if (slices > groups) {
    int64_t perSlice = std::max<int64_t>((totalBytes + slices - 1) / slices + 2048, need);
    plan.groupBytes = (int32_t)(std::min<int64_t>(perSlice, 65536) & ~15);
  }
  plan.treeSlices = (int32_t)std::max<int64_t>(1, slices);
  return plan;
}

} // namespace

namespace {
LaunchPlan ChooseScalarPlan(const Forest &forest, int64_t batchSize, const GPUAutoScheduleOptions *ov,
                            const DeviceLimits &limits, int tileSize, bool peelWalks);
// LDS bytes a tree group must offer the biggest tree of a tiled forest (the null leaf tile and the alignment
// pad of a group included).
int64_t TiledGroupNeed(const Forest &forest, int tileSize) {
  return BiggestTiledTreeBytes(forest, tileSize) + 2 * (int64_t)TileBytes(tileSize) + 16;
}
}

double SlicedWalkMicros(const WalkShape &w, int32_t treeSlices) {
  const int64_t places = (int64_t)w.computeUnits * w.blocksPerUnit, blocks = w.rowBlocks * treeSlices;
  const double share = std::ceil(std::max(1.0, w.groups) / treeSlices) / std::max(1.0, w.groups); // (whole groups)
  double us = 0.0;
  if (const int64_t rounds = blocks / places) // (blocks of later rounds no longer march in step)
    us += (1.0 + 0.88 * (double)(rounds - 1)) * BlockMicros(w, share, w.blocksPerUnit);
  if (const int64_t rest = blocks % places) // the last round: spread over the units, alone on them if they suffice
    us += BlockMicros(w, share, (int)((rest + w.computeUnits - 1) / w.computeUnits));
  return us + (treeSlices > 1 ? kFinalizeMicros : 0.0);
}

double SplitWalkMicros(const WalkShape &w) {
  const double share = (double)w.rowBlocks / ((double)w.computeUnits * w.blocksPerUnit); // of the forest, per block
  // (a part that straddles row blocks stages the rows of each; whole groups only; 3 % for blocks that march in step)
  const double rounded = w.groups > 0 ? std::ceil(share * w.groups) / w.groups : share;
  return BlockMicros(w, rounded * 1.03, w.blocksPerUnit) + std::ceil(share) * BlockMicros(w, 0.0, w.blocksPerUnit) + kFinalizeMicros;
}

namespace {
constexpr int64_t kSmallForestBytes = 24 * 1024;
}

LaunchPlan ChoosePlan(const Forest &forest, int64_t batchSize, const GPUAutoScheduleOptions *ov,
                      const DeviceLimits &limits, const WalkOptions &walk) {
  if (walk.tileSize < 1 || walk.tileSize > kMaxTileSize)
    throw Error("tile size " + std::to_string(walk.tileSize) + " is not supported: the device kernels walk tiles of 1 to " +
                std::to_string(kMaxTileSize) + " nodes");
  if (walk.tileSize > 1 && (int64_t)(forest.numFeatures + 1) * 64 * 4 > 0xFFFF)
    throw Error("tile sizes above 1 need a row tile below 64 KB: " + std::to_string(forest.numFeatures) + " features are too many");
  LaunchPlan wanted;
  wanted.tileSize = walk.tileSize;
  wanted.tiling = walk.tiling;
  LaunchPlan plan = ChooseScalarPlan(forest, batchSize, ov, limits, wanted.WalkTile(), walk.peelWalks);
  plan.tileSize = walk.tileSize;
  plan.tiling = walk.tiling;
  plan.peelWalks = walk.peelWalks;
  plan.deferTails = false;
  if (walk.peelWalks && DeferTailsFit(forest, &plan)) plan.deferTails = true;
  return plan;
}

// Blocks of 1024 lanes, two per compute unit: 256 rows while their tile takes up to 52 KB, else 128 or 64.  A tree group is
// one bundle of two trees for every tree thread, and the trees are cut where that fills the block's half of LDS (a quarter
// more: then some groups are a tree short, and fewer rows are queued).  65536 rows through 40 trees of depth 16 (22000
// nodes each, every child splits again with probability 0.88): 92 us node by node from global memory, 25 here; cut levels
// 7 / 8 / 9 / 10 / 11 27.8 / 27.4 / 26.2 / 24.9 / 29.2, one tree a lane at the same levels 31.2 / 30.2 / 29.0 / 28.0 / 28.1, four
// 25.7 / 25.3 / 26.4 at levels 8 to 10.  70 features: 109 us -> 33 with 128 rows a block (40 with 64), 100 features 133 -> 36,
// 150 features 177 -> 54.
bool ChooseDeepWalk(const Forest &forest, const DeviceLimits &limits, LaunchPlan *plan, std::vector<int32_t> *cuts) {
  if (forest.numClasses > 0 || forest.trees.empty() || forest.numFeatures + 1 >= (1 << kTailFeatureBits)) return false;
  const auto tileBytes = [&](int32_t rows) { return (int64_t)(forest.numFeatures + 1) * rows * 4; };
  int32_t rows = 256;
  while (rows > 64 && tileBytes(rows) > 52 * 1024) rows /= 2;
  *plan = LaunchPlan();
  plan->rowsPerBlock = rows;
  plan->treeThreads = 1024 / rows;
  plan->interleave = 2;
  plan->deferTails = true;
  const int64_t queues = (int64_t)(plan->ThreadsPerBlock() / 64) * kDeferBytesPerWave;
  const int64_t room = std::min<int64_t>(65536, limits.ldsBytesPerBlock / 2 - tileBytes(rows) - queues - 1024);
  const int64_t bundles = (int64_t)plan->treeThreads * plan->interleave;
  const int64_t mostTop = std::min(room * 5 / 4 / bundles, room) / kNodeBytes - 4;
  if (mostTop < 31) return false;
  int64_t tails = 1; // places of the tail array: the null leaf, the cut levels' internal nodes and all below them
  cuts->clear();
  for (const Tree &tree : forest.trees) {
    int64_t top = 0;
    int32_t depth = 0, cut = -1;
    std::vector<int32_t> level{0}, below;
    for (; !level.empty(); ++depth) {
      if (cut < 0 && top + (int64_t)level.size() > mostTop) {
        cut = depth - 1;
        tails += (int64_t)level.size() / 2; // (the parents of this level)
      }
      (cut < 0 ? top : tails) += (int64_t)level.size();
      below.clear();
      for (int32_t n : level) {
        if (tree.IsLeaf(n)) continue;
        below.push_back(tree.left[n]);
        below.push_back(tree.right[n]);
      }
      level.swap(below);
    }
    cuts->push_back(cut < 0 ? depth - 1 : cut);
  }
  if (tails > kMaxTailNodes) return false;
  plan->groupBytes = (int32_t)(std::min<int64_t>(room, std::max<int64_t>((bundles * mostTop + 4) * kNodeBytes, 1024)) & ~15);
  return true;
}

// One round of blocks.  More slices (each stages the rows again) took 30 us with 4 and 34 with 5 where 2 take 25, one 28.
int32_t DeepWalkSlices(int64_t rowBlocks, int64_t groups, const DeviceLimits &limits) {
  return (int32_t)std::max<int64_t>(1, std::min<int64_t>(2LL * limits.computeUnits / std::max<int64_t>(1, rowBlocks), groups));
}

bool SmallForestBlocks(const Forest &forest, const LaunchPlan &plan) {
  return plan.rowsPerBlock == 128 && plan.treeThreads == 4 && (int64_t)forest.NumNodes() * kNodeBytes <= kSmallForestBytes;
}

bool DeferTailsFit(const Forest &forest, LaunchPlan *plan) {
  if (plan->kernel != LaunchPlan::Kernel::kRowParallelLds || plan->WalkTile() != 1 || plan->quantizedRows || plan->rankRows16 ||
      plan->featureOffsetInWords || forest.numClasses > 0)
    return false;
  // Blocks of small forests walk whole trees faster: 45 skewed forests of 2 to 24 KB, rows along the spines, 12000 to 950000 rows,
  // 4 % (30 trees of depth 9) to 20 % (17 trees of depth 8, 610597 rows 32.3 -> 25.8 us) in 128 x 4, and all of them than with
  // deferred tails in 256 x 4.
  if (SmallForestBlocks(forest, *plan)) return false;
  // every wave's queue comes out of the tree group's share of LDS
  const int64_t extra = (int64_t)(plan->ThreadsPerBlock() / 64) * kDeferBytesPerWave + 32;
  if (forest.numFeatures + 1 >= (1 << kTailFeatureBits)) return false;
  const int64_t need = (BiggestTreeNodes(forest) + 2) * kNodeBytes;
  if (plan->groupBytes - extra < std::max<int64_t>(need, 8192)) return false;
  plan->groupBytes = (int32_t)((plan->groupBytes - extra) & ~15);
  return true;
}

namespace {

// tileSize > 1 (tiles chosen by a profile): the plan must be the row-parallel kernel on f32 rows with byte offsets (tiles hold byte offsets
// into a row tile below 64 KB), and groups are sized for tiles, which take three to eight times the bytes of
// scalar nodes.
LaunchPlan ChooseScalarPlan(const Forest &forest, int64_t batchSize, const GPUAutoScheduleOptions *ov,
                            const DeviceLimits &limits, int tileSize, bool peelWalks) {
  if (tileSize > 1) {
    const int64_t need = TiledGroupNeed(forest, tileSize);
    if (need > 65536)
      throw Error("tile sizes above 1 need every tree to fit one LDS tree group; this forest has a tree that does not");
    LaunchPlan plan;
    plan.kernel = LaunchPlan::Kernel::kRowParallelLds;
    int32_t rb = 256;
    if (ov && ov->numRowsPerTB > 0) rb = std::max(64, std::min(256, FloorPow2(ov->numRowsPerTB)));
    // two blocks per CU while 24 KB remain for a group, byte offsets below 64 KB
    auto tileBytes = [&](int32_t r) { return (int64_t)(forest.numFeatures + 1) * r * 4; };
    while (rb > 64 && (tileBytes(rb) > 0xFFFF || limits.ldsBytesPerBlock / 2 - tileBytes(rb) < 24 * 1024)) rb /= 2;
    plan.rowsPerBlock = rb;
    plan.treeThreads = std::max(1, 1024 / rb);
    if (ov && ov->numTreeThreads > 0) plan.treeThreads = std::max(1, std::min(ov->numTreeThreads, 1024 / rb));
    plan.interleave = 2;
    if (ov && ov->treeWalkInterleaveFactor > 0) plan.interleave = std::min(4, FloorPow2(ov->treeWalkInterleaveFactor));
    const int64_t meet = forest.numClasses > 0 ? (int64_t)rb * plan.treeThreads * 8 : 0;
    int64_t budget = limits.ldsBytesPerBlock / 2;
    int64_t group = std::min<int64_t>(65536, budget - tileBytes(rb) - meet - 512);
    if (group < need) group = std::min<int64_t>(65536, limits.ldsBytesPerBlock - tileBytes(rb) - meet - 512);
    group = std::min<int64_t>(group, 256LL * rb * plan.treeThreads);
    if (group < need) throw Error("the biggest tree does not fit LDS next to the row tile when tiled");
    plan.groupBytes = (int32_t)(group & ~15);
    const int64_t rowBlocks = std::max<int64_t>(1, (batchSize + rb - 1) / rb);
    const int64_t totalBytes = (int64_t)forest.NumNodes() * (tileSize > kMaxSelectTile ? 40 : 24);
    int64_t slices = 1;
    const int64_t wantBlocks = 2LL * limits.computeUnits;
    if (rowBlocks < wantBlocks) slices = (wantBlocks + rowBlocks - 1) / rowBlocks;
    slices = std::min<int64_t>(slices, std::max<int64_t>(1, totalBytes / plan.groupBytes));
    plan.treeSlices = (int32_t)std::max<int64_t>(1, slices);
    return plan;
  }
  // A tree that cannot sit in one LDS group walks from global memory; so do rows that neither LDS form can
  // hold (below): more than 16383 features have no 16-bit byte offset inside one row-major LDS row.
  auto globalPlan = [&]() {
    LaunchPlan plan;
    plan.kernel = LaunchPlan::Kernel::kGlobalWalk;
    plan.rowsPerBlock = 256;
    plan.interleave = 4;
    if (ov && ov->treeWalkInterleaveFactor > 0)
      plan.interleave = std::min(kMaxInterleave, FloorPow2(ov->treeWalkInterleaveFactor));
    const int64_t rowBlocks = std::max<int64_t>(1, (batchSize + 255) / 256);
    int64_t slices = 1;
    if (rowBlocks < 4LL * limits.computeUnits) slices = (4LL * limits.computeUnits + rowBlocks - 1) / rowBlocks;
    plan.treeSlices = (int32_t)std::max<int64_t>(1, std::min<int64_t>(slices, (int64_t)forest.trees.size()));
    plan.groupBytes = 0;
    return plan;
  };
  if ((BiggestTreeNodes(forest) + 2) * kNodeBytes > 65536) return globalPlan();
  const bool rowMajorFits = (int64_t)(forest.numFeatures + 1) * 4 <= 0xFFFF &&
                            (int64_t)(forest.numFeatures + 1) * 4 + (BiggestTreeNodes(forest) + 2) * kNodeBytes + 4096 <=
                                limits.ldsBytesPerBlock;
  bool fitsTransposed = false;
  {
    bool words = false;
    fitsTransposed = RowTileFits(forest.numFeatures, 64, limits.ldsBytesPerBlock, &words);
  }
  if (batchSize > 0 && batchSize <= 128 && rowMajorFits) return ChooseTreeParallelPlan(forest, batchSize, ov, limits);
  if (!fitsTransposed) {
    // Rows too wide for 64 f32 rows in LDS: one-byte ranks (exact) if every feature has few enough
    // distinct thresholds and 64 rank rows fit; otherwise a few f32 rows with several lanes each.
    const int64_t tile = (int64_t)(forest.numFeatures + 1) * 64;
    const int64_t need = (BiggestTreeNodes(forest) + 2) * kNodeBytes;
    const int64_t room = limits.ldsBytesPerBlock - tile - 2048 - (forest.numClasses > 0 ? 1024 * 8 : 0);
    if (room >= std::max<int64_t>(need, 8192) && forest.numFeatures * 16 <= 0xFFFF &&
        MaxThresholdsPerFeature(forest) <= 254) {
      LaunchPlan plan;
      plan.kernel = LaunchPlan::Kernel::kRowParallelLds;
      plan.quantizedRows = true;
      plan.rowsPerBlock = 64;
      plan.treeThreads = 16;
      if (ov && ov->numTreeThreads > 0) plan.treeThreads = std::max(1, std::min(ov->numTreeThreads, 16));
      plan.interleave = 2;
      if (ov && ov->treeWalkInterleaveFactor > 0)
        plan.interleave = std::min(kMaxInterleave, FloorPow2(ov->treeWalkInterleaveFactor));
      plan.groupBytes = (int32_t)(std::min<int64_t>({room, 65536, 256LL * plan.ThreadsPerBlock()}) & ~15);
      const int64_t rowBlocks = std::max<int64_t>(1, (batchSize + 63) / 64);
      const int64_t totalBytes = (int64_t)forest.NumNodes() * kNodeBytes;
      int64_t slices = 1;
      if (rowBlocks < limits.computeUnits) slices = (limits.computeUnits + rowBlocks - 1) / rowBlocks;
      slices = std::min<int64_t>(slices, std::max<int64_t>(1, totalBytes / plan.groupBytes));
      plan.treeSlices = (int32_t)std::max<int64_t>(1, slices);
      return plan;
    }
    return rowMajorFits ? ChooseTreeParallelPlan(forest, batchSize, ov, limits) : globalPlan();
  }

  LaunchPlan plan;
  plan.kernel = LaunchPlan::Kernel::kRowParallelLds;

  // Block shape, from timings on MI355X (blocks of 1024 lanes; 600-1000 trees of depth 6-8; 28..520 features).
  // Two blocks per CU hide each other's group loads and barriers, but only while enough LDS is left for
  // the tree groups; a narrower row tile buys bigger groups; past that one block per CU with the biggest
  // groups wins.  In order of preference:
  //   256 rows x 4 tree threads, two blocks per CU, while >= 16 KB remain for a group   (up to ~60 features)
  //   128 x 8, two blocks, while >= 20 KB remain                                        (up to ~118)
  //    64 x 16, two blocks, while >= 40 KB remain                                       (up to ~155)
  //   128 x 8, one block, while >= 56 KB remain                                         (up to ~195)
  //    64 x 16, one block                                                               (as long as the tile fits)
  const int32_t halfLds = limits.ldsBytesPerBlock / 2;
  bool words = false;
  auto treeThreadsFor = [&](int32_t r) {
    int32_t tt = std::max(1, 1024 / r);
    if (ov && ov->numTreeThreads > 0) tt = std::max(1, std::min(ov->numTreeThreads, 1024 / r));
    return tt;
  };
  // LDS left for a tree group beside the row tile (and the classifiers' meeting area)
  auto roomFor = [&](int32_t r, int32_t ldsBytes) -> int64_t {
    const int64_t tile = (int64_t)(forest.numFeatures + 1) * r * 4;
    const int64_t meetBytes = forest.numClasses > 0 ? (int64_t)r * treeThreadsFor(r) * 8 : 0;
    return (int64_t)ldsBytes - tile - meetBytes - 512;
  };
  int32_t rb = 64;
  int32_t budget = limits.ldsBytesPerBlock;
  if (ov && ov->numRowsPerTB > 0) { // the caller's block shape: two blocks per CU if 16 KB remain, else one
    rb = std::max(64, FloorPow2(ov->numRowsPerTB));
    while (rb > 64 && roomFor(rb, limits.ldsBytesPerBlock) < 16384) rb /= 2;
    if (roomFor(rb, halfLds) >= 16384) budget = halfLds;
  } else if (roomFor(256, halfLds) >= 16384) {
    rb = 256, budget = halfLds;
  } else if (roomFor(128, halfLds) >= 20480) {
    rb = 128, budget = halfLds;
  } else if (roomFor(64, halfLds) >= 40960) {
    rb = 64, budget = halfLds;
  } else if (roomFor(128, limits.ldsBytesPerBlock) >= 57344) {
    rb = 128;
  }
  if (!RowTileFits(forest.numFeatures, rb, budget, &words))
    throw Error("row tile of " + std::to_string(forest.numFeatures) + " features does not fit LDS");
  plan.rowsPerBlock = rb;
  plan.featureOffsetInWords = words;
  plan.treeThreads = treeThreadsFor(rb);

  plan.interleave = 4;
  if (ov && ov->treeWalkInterleaveFactor > 0)
    plan.interleave = std::min(kMaxInterleave, FloorPow2(ov->treeWalkInterleaveFactor));

  const int64_t rowTile = (int64_t)(forest.numFeatures + 1) * rb * 4;
  const int64_t need = (BiggestTreeNodes(forest) + 2) * kNodeBytes;
  if (need > 65536) throw Error("a tree does not fit one LDS tree group");
  const int64_t meet = forest.numClasses > 0 ? (int64_t)rb * plan.treeThreads * 8 : 0; // cross-wave pass
  // (LDS is handed out in coarse pieces: leave slack or the second block will not fit)
  int64_t group = std::min<int64_t>(65536, budget - rowTile - meet - 512);
  if (group < need) group = std::min<int64_t>(65536, limits.ldsBytesPerBlock - rowTile - meet - 512);
  group = std::min<int64_t>(group, 256LL * rb * plan.treeThreads); // 16 prefetch registers of 16 bytes per lane
  if (group < need) throw Error("the biggest tree does not fit LDS next to the row tile");
  plan.groupBytes = (int32_t)(group & ~15);

  // Tree slices: when the batch alone cannot fill the chip, blocks share a row
  // tile and split the tree groups between them.
  const int64_t rowBlocks = std::max<int64_t>(1, (batchSize + rb - 1) / rb);
  const int64_t totalBytes = (int64_t)forest.NumNodes() * kNodeBytes;
  int64_t groups = std::max<int64_t>(1, (totalBytes + plan.groupBytes - 1) / plan.groupBytes);
  int64_t slices = 1;
  if (rowBlocks < 2LL * limits.computeUnits) {
    WalkShape shape;
    shape.rowBlocks = rowBlocks;
    shape.rowsPerBlock = rb;
    shape.numFeatures = forest.numFeatures;
    for (const Tree &tree : forest.trees) shape.levels += tree.Depth();
    shape.computeUnits = limits.computeUnits;
    shape.blocksPerUnit = budget == halfLds ? 2 : 1;
    double best = 0.0;
    // (at least 16 KB of trees per slice)
    for (int64_t s = 1; s <= std::min<int64_t>(64, std::max<int64_t>(1, totalBytes / 16384)); ++s) {
      shape.groups = (double)std::max<int64_t>(groups, s);
      double us = SlicedWalkMicros(shape, (int32_t)s);
      if (rowBlocks * s > shape.computeUnits * shape.blocksPerUnit) us = std::min(us, SplitWalkMicros(shape)); // (as the launch will choose)
      if (s == 1 || us < best) best = us, slices = s;
    }
  }
  // Smaller row blocks than two blocks per compute unit leave room for:
  //  * up to a block of 256 rows for each compute unit, and too few trees to slice: 128 rows x 8 tree threads, two of which share a
  //    unit once every other unit would have a block of 256.  Up to there they always win or tie (20761 rows x 266 trees of depth
  //    6 21.0 -> 13.4 us, 8017 x 61 7.5 -> 7.0, 20755 x 79 of depth 3 7.0 and 7.1).  Beyond, twice the blocks stage every group:
  //    that pays where the rows' walk is long for the groups there are, or where the smaller row tile saves groups.  125 forests of
  //    30 to 320 trees on 32800 to 65536 rows, levels of a walk, groups beside 256 rows and beside 128: 541 levels 1 and 1 groups
  //    10.5 -> 9.6 us, 481 1 1 9.8 -> 9.3, 403 1 1 8.9 and 8.6, 340 1 1 7.9 and 8.4, 258 1 1 7.4 -> 8.1; 700 2 2 12.6 -> 12.1, 572 2 2
  //    12.4 and 12.8, 561 2 2 11.3 -> 12.0; 632 3 3 (of 33 features) 14.4 -> 13.5, 650 3 3 (of 6) 12.8 and 13.1; 700 4 4 15.5 ->
  //    14.8; 397 2 1 9.7 -> 8.9.  Taken of them: none that loses, left: none that would gain more than 0.4 us;
  //  * forests of up to 24 KB, whose rows take as long to stage as to walk: 128 x 4, of which three and more to a unit take
  //    turns.  2^20 rows x 60 trees of depth 5 69.6 -> 58.0 us, 210411 x 62 19.6 -> 17.2, 402162 x 51 of depth 4 30.0 -> 26.0
  //    (29 KB: 37.7 and 38.5).  Four to a unit, that is: of 89 forests of 2 to 24 KB on 131100 to 2^20 rows they win by 0 to 16 %
  //    where four fit its LDS (but for one, 1 %), and where three do lose 2 to 9 % (388783 rows x 60 trees of 58 features 31.9 ->
  //    34.7 us, 311105 x 17 of 51 25.0 -> 27.7) unless one round of either is enough (157757 rows 12.8 -> 12.3, 199341 29.9 -> 29.2).
  // (Not where the biggest tree asks for more than the group beside them: the blocks of 256 rows may have taken the whole LDS for it.)
  if (forest.numClasses == 0 && slices == 1 && rb == 256 && budget == halfLds && roomFor(128, halfLds) >= need &&
      !(ov && (ov->numRowsPerTB > 0 || ov->numTreeThreads > 0))) {
    const int64_t smaller = std::min<int64_t>(65536, roomFor(128, halfLds)) & ~15LL;
    const int64_t smallerGroups = std::max<int64_t>(1, (totalBytes + smaller - 1) / smaller);
    int64_t levels = 0;
    for (const Tree &tree : forest.trees) levels += tree.Depth();
    const bool fewTrees = totalBytes <= kSmallForestBytes;
    const int64_t enough = groups == 1 ? 390 : 670 - forest.numFeatures * 6 / 5 - 240 * (groups - smallerGroups);
    const bool idle = rowBlocks * 2 <= limits.computeUnits || (rowBlocks <= limits.computeUnits && (fewTrees || levels >= enough));
    const bool fourFit = (int64_t)(forest.numFeatures + 1) * 128 * 4 + totalBytes + 32 <= limits.ldsBytesPerBlock / 4;
    if (idle || (fewTrees && rowBlocks > 2LL * limits.computeUnits && (fourFit || rowBlocks <= 5LL * limits.computeUnits / 2))) {
      rb = plan.rowsPerBlock = 128;
      plan.treeThreads = fewTrees ? 4 : 8;
      plan.groupBytes = (int32_t)(fewTrees ? std::min<int64_t>(smaller, totalBytes + 1024) & ~15LL : smaller);
    }
  }
  if (slices > groups) { // more, smaller groups so that every slice has one
    int64_t perSlice = std::max<int64_t>((totalBytes + slices - 1) / slices + 4096, need);
    if (perSlice < plan.groupBytes) plan.groupBytes = (int32_t)((perSlice + 15) & ~15);
  }
  // Four trees side by side hide more latency than two, but where a group holds fewer trees than the tree threads could take
  // that way, threads without a bundle wait for the others.  262144 rows, 200 to 300 trees, two and four trees a lane: four tree
  // threads 54 features 16.2 trees a group 132 and 122 us, 14.0 146 and 142, 12.1 106 and 120; eight 27.9 136 and 126, 22.8 147
  // and 148, 19.5 158 and 171, 8.0 207 and 246; sixteen 47 147 and 141, 40 161 and 161, 31 183 and 189, 12 242 and 282; 40000
  // rows alike.  (One tree a lane is never faster.)  Classifiers alike, but sixteen tree threads 16.9 298 and 279, 20.1 2396 and
  // 2268, 23.2 105 and 105, 25.4 133 and 138, 80 and 83: a group holds few classes at a time.
  const double fewInGroup = forest.numClasses > 0 ? std::min(24.0, 2.4 * plan.treeThreads + 3.4) : 2.4 * plan.treeThreads + 3.4;
  // Groups end on whole rounds of the tree threads, so that bundles of two can take more of them.  Not where the slices then have half
  // as many again to walk: one group and two 12708 rows x 89 trees in ten slices 10.8 -> 11.9 us, 16925 x 72 in seven 10.8 -> 11.5,
  // two and three 4814 x 193 in five 10.2 -> 11.3, 15744 x 80 in four 10.6 -> 10.9; three and four 11.8 and 11.5, 14.8 and 15.0,
  // five and six 19.8 -> 19.0, 14.9 -> 14.2, alike 13.2 -> 12.1.
  plan.treeSlices = (int32_t)std::max<int64_t>(1, slices);
  // As it will be packed: deferred tails keep all leaves in LDS, peeled walks without them need not.  Three classes, trees of depth 8, two
  // trees a lane (what counting whole trees asks for) and four: 30000 rows x 61 trees of 33 features 15.6 and 13.1 us, 2^18 x 161 79.9 and
  // 73.4, 2^20 x 89 190 and 170, 2^18 x 89 of 57 features 79.0 and 72.9; but 2^18 x 61 of 130 features 112.5 and 117.4.
  LaunchPlan walked = plan, queued = plan;
  walked.deferTails = peelWalks && DeferTailsFit(forest, &queued);
  const int64_t inLds = LeavesOutside(forest, walked) ? TreeBytesInLds(forest, true) : totalBytes;
  if (!(ov && ov->treeWalkInterleaveFactor > 0) && (double)plan.groupBytes * (double)forest.trees.size() < fewInGroup * (double)inLds) {
    LaunchPlan two = walked;
    two.interleave = 2;
    const auto turns = [&](const LaunchPlan &p) { return (CountTreeGroups(forest, p) + slices - 1) / slices; };
    if (slices == 1 || (forest.numClasses > 1 && PacksOwnClasses(forest, two)) || turns(two) * 2 < turns(walked) * 3) plan.interleave = 2;
  }
  // Classes of the tree threads' own (PackForest) need groups of a bundle for every tree thread: bundles of two where four do
  // not fit, that way costs less (the packer's costs), and the packer will take it: where it does not, two side by side lose (607
  // trees, 13 classes, 189139 rows 235 and 247 us, 321 trees, 7 classes, 2642 rows 27.2 and 29.2).  200000 rows, four and two side by side: 100 trees of depth 7, 90
  // features, 10 classes 103.7 and 60.7 us; 300 of depth 8, 54 features, 12 classes 177.1 and 137.8; 200 of depth 8, 70
  // features, 6 classes 132.8 and 105.9; 400 of depth 7, 90 features, 8 classes 195.4 and 152.3.
  if (forest.numClasses > 1 && plan.treeThreads > 1 && plan.interleave == 4 && !(ov && ov->treeWalkInterleaveFactor > 0) &&
      (double)plan.groupBytes * (double)forest.trees.size() < (4.0 * std::min(plan.treeThreads, forest.numClasses) + 0.3) * (double)inLds) {
    double levels = 0.0;
    for (const Tree &tree : forest.trees) levels += tree.Depth();
    levels /= (double)forest.trees.size();
    const double ofClass = (double)forest.trees.size() / forest.numClasses, threads = plan.treeThreads;
    const double own = std::ceil(forest.numClasses / threads) * std::ceil(ofClass / 2) * 2 * levels;
    LaunchPlan two = plan;
    two.interleave = 2;
    if (own < forest.numClasses * (std::ceil(ofClass / (4 * threads)) * 4 * levels + 20.0) && PacksOwnClasses(forest, two)) plan.interleave = 2;
  }
  // Tree threads with classes of their own never meet: their place behind the rows goes to the groups (2^20 rows x 54 features, 800
  // trees of depth 6, 8 classes: 25 groups and 17, 778 -> 741 us; 65537 rows with sums 81.6 -> 79.7).  The packer takes it where it
  // finds the classes to be theirs.
  if (meet > 0 && plan.groupBytes == (int32_t)(group & ~15)) {
    const int32_t roomy = (int32_t)(std::min<int64_t>({group + meet, 65536, 256LL * plan.ThreadsPerBlock()}) & ~15);
    if (forest.numClasses > 1 && plan.treeThreads > 1 && roomy > plan.groupBytes) plan.ownGroupBytes = roomy;
  }
  return plan;
}

} // namespace

void SeparateGroupSizes(const Forest &forest, const HitCountProfile *profile, const DeviceLimits &limits, LaunchPlan *plan) {
  if (forest.numClasses < 2 || plan->kernel != LaunchPlan::Kernel::kRowParallelLds) return;
  const PackedModel pm = PackForest(forest, *plan, profile); // (which refuses what a damaged file may hold)
  if (!pm.ownClasses) return;
  const int64_t place = plan->ThreadsPerBlock() * 8, need = (BiggestTreeNodes(forest) + 2) * kNodeBytes;
  for (const int64_t budget : {limits.ldsBytesPerBlock / 2, limits.ldsBytesPerBlock}) { // (the planner's)
    const int64_t room = budget - (int64_t)pm.RowTileBytes() - 512;
    if (plan->groupBytes > room) continue;
    const int64_t beside = (room - place) & ~15LL;
    if (beside >= plan->groupBytes || beside < std::max<int64_t>(need, 1024)) return;
    plan->ownGroupBytes = plan->groupBytes;
    plan->groupBytes = (int32_t)beside;
    return;
  }
}

std::vector<LaunchPlan> CandidatePlans(const Forest &forest, int64_t batchSize, const DeviceLimits &limits,
                                       const WalkOptions &walk) {
  std::vector<LaunchPlan> out;
  LaunchPlan base = ChoosePlan(forest, batchSize, nullptr, limits, walk);
  out.push_back(base);
  if (base.WalkTile() > 1) { // block shapes and interleave factors of the tiled walk
    for (int32_t rb : {64, 128, 256})
      for (int32_t k : {1, 2, 4}) {
        LaunchPlan p = base;
        p.rowsPerBlock = rb;
        p.treeThreads = 1024 / rb;
        p.interleave = k;
        const int64_t tile = (int64_t)(forest.numFeatures + 1) * rb * 4;
        if (tile > 0xFFFF) continue;
        const int64_t meet = forest.numClasses > 0 ? (int64_t)rb * p.treeThreads * 8 : 0;
        int64_t group = std::min<int64_t>(65536, limits.ldsBytesPerBlock / 2 - tile - meet - 2048);
        if (group < TiledGroupNeed(forest, base.WalkTile())) continue;
        if (base.treeSlices > 1) group = std::min<int64_t>(group, base.groupBytes);
        p.groupBytes = (int32_t)(group & ~15);
        bool dup = false;
        for (auto &q : out)
          dup = dup || (q.rowsPerBlock == p.rowsPerBlock && q.interleave == p.interleave && q.groupBytes == p.groupBytes);
        if (!dup) out.push_back(p);
      }
    return out;
  }
  if (base.kernel == LaunchPlan::Kernel::kGlobalWalk) {
    for (int32_t k : {1, 2, 8}) {
      LaunchPlan p = base;
      p.interleave = k;
      out.push_back(p);
    }
    return out;
  }
  if (base.kernel == LaunchPlan::Kernel::kTreeParallel) {
    for (int32_t lanes : {base.treeLanes / 2, base.treeLanes * 2})
      for (int32_t k : {1, 2}) {
        LaunchPlan p = base;
        p.treeLanes = lanes;
        p.interleave = k;
        if (lanes < 1 || p.ThreadsPerBlock() > 1024 || p.ThreadsPerBlock() % 64 != 0) continue;
        if (lanes < 64 && 64 % lanes != 0) continue;
        out.push_back(p);
      }
    return out;
  }
  const int64_t need = (BiggestTreeNodes(forest) + 2) * kNodeBytes;
  for (int32_t rb : {64, 128, 256, 512})
    for (int32_t tt : {1, 2, 4, 8, 16})
      for (int32_t k : {2, 4, 8})
        for (int blocksPerCu : {1, 2, 3, 4, 6, 8}) {
          if (rb * tt > 1024 || rb * tt * blocksPerCu > 2048) continue; // (a compute unit holds 32 waves)
          bool words = false;
          const int32_t budget = limits.ldsBytesPerBlock / blocksPerCu;
          if (!RowTileFits(forest.numFeatures, rb, budget + 8192, &words)) continue;
          LaunchPlan p = base;
          p.rowsPerBlock = rb;
          p.treeThreads = tt;
          p.ownGroupBytes = 0; // (what its groups may take is said below)
          p.featureOffsetInWords = words;
          p.interleave = k;
          const int64_t rowTile = (int64_t)(forest.numFeatures + 1) * rb * 4;
          int64_t group = std::min<int64_t>(65536, budget - rowTile - (forest.numClasses > 0 ? (int64_t)rb * tt * 8 : 0) - 2048);
          group = std::min<int64_t>(group, 256LL * rb * tt); // 16 prefetch registers of 16 bytes per lane
          if (group < need || group < 8192) continue;
          if (base.treeSlices > 1) group = std::min<int64_t>(group, base.groupBytes);
          p.groupBytes = (int32_t)(group & ~15);
          if (base.deferTails) {
            p.deferTails = false;
            if (!DeferTailsFit(forest, &p)) continue;
            p.deferTails = true;
          }
          bool dup = false;
          for (auto &q : out)
            dup = dup || (q.rowsPerBlock == p.rowsPerBlock && q.treeThreads == p.treeThreads &&
                          q.interleave == p.interleave && q.groupBytes == p.groupBytes);
          if (!dup) out.push_back(p);
        }
  // Two-byte rank rows (a ranking kernel in front of the walk, half the row tile): the timed search counts both
  // kernels, so the form is kept only where the walk gains more than the ranking costs.
  if (!base.quantizedRows && base.treeSlices == 1)
    for (int32_t rb : {256, 512}) {
      const int64_t rowTile = (int64_t)((forest.numFeatures + 2) / 2) * rb * 4;
      if (rowTile > 0xFFFF) continue;
      LaunchPlan p = base;
      p.rankRows16 = true;
      p.deferTails = false;
      p.featureOffsetInWords = false;
      p.rowsPerBlock = rb;
      p.treeThreads = 1024 / rb;
      p.ownGroupBytes = 0;
      p.interleave = 4;
      int64_t group = std::min<int64_t>(65536, limits.ldsBytesPerBlock / 2 - rowTile - (forest.numClasses > 0 ? 1024 * 8 : 0) - 2048);
      if (group < need || group < 8192) continue;
      p.groupBytes = (int32_t)(group & ~15);
      out.push_back(p);
    }
  return out;
}

} // namespace tbamd
