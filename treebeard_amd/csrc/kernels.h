// Host-callable launchers of the HIP kernels (kernels.hip).
#pragma once

#include "device_model.h"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace tbamd {

// Scalars of the row-parallel walk (passed by value, live in SGPRs).
struct WalkScalars {
  int64_t rows = 0;
  int32_t numFeatures = 0;
  int32_t numClasses = 0;
  int32_t numGroups = 0;
  int32_t treeSlices = 1;
  uint32_t groupRegionBytes = 0; // LDS bytes reserved for one tree group (multiple of 16)
  int32_t transform = 0;         // 0 identity, 1 sigmoid
  int32_t numTrees = 0;
  int32_t rowsPerBlock = 0;      // rows per block (both kernels)
  int32_t treeThreads = 1;       // row-parallel kernel: lanes (in different waves) that share a row
  int32_t treeLanes = 1;         // tree-parallel kernel: lanes per row (power of two)
  // Row-parallel kernels, classifiers with one tree slice: the kernel keeps the running arg-max of the class
  // sums (which arrive in ascending class order) and stores the class id itself; no partial sums, no finalize.
  int32_t fuseArgmax = 0;
  // Row-parallel scalar walk of a classifier: bundle i of a group is tree thread i % treeThreads', and class c's trees are all
  // tree thread c % treeThreads' (PackedModel::ownClasses).
  int32_t ownClasses = 0;
  // Scalar row-parallel walk: the leaves of a bundle's last level are not in LDS (PackedModel::leavesOutside).
  int32_t leavesOutside = 0;
  // Scalar row-parallel walk on an f32 tile with byte offsets: trees may end in stubs (device_model.h); the row
  // tile then has a column for the stub feature and every wave a queue of deferred walks behind it.
  int32_t deferTails = 0;
  int32_t tailDepth = 0;         // steps the deepest deferred walk takes below its stub
  int32_t tileHops = 1;          // eight-slot tiles: links a tile step follows at most (levels of nodes inside a tile)
  double initialValue = 0.0;
};

struct WalkParams {
  WalkScalars s;
  const float *x = nullptr;       // rows x numFeatures, row-major, device
  const uint4 *nodes16 = nullptr; // packed nodes viewed as 16-byte pieces
  const DeviceBundle *bundles = nullptr;
  const DeviceNode *bundleRoots = nullptr; // interleave root-node copies per bundle (row-parallel f32 walk)
  const DeviceGroup *groups = nullptr;
  const DeviceNode *tailNodes = nullptr;   // deferred tails: the subtrees below the stubs (PackedModel::tailNodes)
  const int32_t *tailOrigin = nullptr;     // ... and their original node ids (leaf-id dump)
  const DeviceGlobalNode *globalNodes = nullptr; // global-memory walk only
  const DeviceGlobalTree *globalTrees = nullptr;
  bool peelWalks = false;         // tiled walk: bundles carry peel depths below their depths
  // Row-parallel scalar walk: tree groups go straight from global memory into LDS (no staging registers); the
  // block waits for its copy, so this pays when a second block on the CU walks meanwhile.
  bool directStaging = false;
  float *out = nullptr;           // used when the epilogue is fused (1 slice; class ids as float32 with fuseArgmax)
  int8_t *classOut = nullptr;     // fuseArgmax: class ids as int8 (out is then null)
  double *partial = nullptr;      // [partials][rows][max(1, classes)] otherwise
  // leaf-id dump (parity checks only)
  int32_t *leafIds = nullptr;     // [rows][numTrees]
  const int32_t *nodeOrigin = nullptr;
  const int32_t *slotTree = nullptr;
  hipEvent_t done = nullptr;      // recorded when this kernel completes
  // Row-parallel walk on f32 or one-byte rank rows: `splitBlocks` blocks (0: one per row block and
  // tree slice) share the units row block x tree group evenly; partial holds SplitLine::Slots slots.
  int32_t splitBlocks = 0;
};

// Row blocks x tree groups as one line of units, cut into equal parts for `blocks` <= units blocks.
struct SplitLine {
  int64_t units;
  int32_t groups, blocks;
#if defined(__HIP__)
  __host__ __device__
#endif
  int64_t FirstUnit(int64_t block) const { return block * units / blocks; }
#if defined(__HIP__)
  __host__ __device__
#endif
  int64_t FirstBlock(int64_t rowBlock) const { return ((rowBlock * groups + 1) * blocks - 1) / units; } // (the owner of its first unit)
#if defined(__HIP__)
  __host__ __device__
#endif
  int Parts(int64_t rowBlock) const { return (int)(((rowBlock + 1) * groups * blocks - 1) / units - FirstBlock(rowBlock)) + 1; }
  // The most parts any row block has.
  static int64_t Slots(int64_t blocks, int64_t rowBlocks) { return (blocks + rowBlocks - 1) / rowBlocks + (blocks % rowBlocks ? 1 : 0); }
};

struct FinalizeParams {
  double *partial = nullptr;   // [slices][rows][max(1, classes)]
  int64_t rows = 0;
  int32_t numClasses = 0;
  int32_t treeSlices = 1;      // number of partial sums per (row, class)
  int32_t splitBlocks = 0;     // a split walk: its blocks, rows per block and tree groups (treeSlices: slots)
  int32_t rowsPerBlock = 0, groups = 0;
  double initialValue = 0.0;
  int32_t transform = 0;
  float *out = nullptr;        // regression / binary prediction, may be null for multiclass
  int8_t *classOut = nullptr;  // multiclass: arg-max class id
  float *margins = nullptr;    // optional [rows][classes] per-class sums
  float *probabilities = nullptr; // optional [rows][classes] softmax
  hipEvent_t done = nullptr;
};

// Batches of a few rows: one launch that also finishes (no partial sums, no finalize kernel).
struct FewRowsParams {
  const float *x = nullptr;                   // rows x numFeatures, row-major; device memory or pinned host memory
  const DeviceFewRowsBlock *blocks = nullptr; // PackFewRows
  const int32_t *classBegin = nullptr;
  int64_t rows = 0;
  int32_t numFeatures = 0, numTrees = 0, numClasses = 0;
  int32_t transform = 0;
  double initialValue = 0.0;
  float *out = nullptr;                       // as in FinalizeParams
  int8_t *classOut = nullptr;
  float *margins = nullptr;
  float *probabilities = nullptr;
  hipEvent_t done = nullptr;
};

// How LaunchFewRows cuts a batch.
struct FewRowsShape {
  int rowsPerBlock, threads;
  size_t leafStride, ldsBytes; // floats per tree in the leaf array; LDS of a block
};
constexpr size_t kFewRowsLds = 64 * 1024;
inline FewRowsShape ShapeOfFewRows(int64_t rows, int numFeatures, int numTrees, int numClasses) {
  FewRowsShape s;
  s.rowsPerBlock = (int)std::max<int64_t>(1, (rows + 255) / 256); // a block per compute unit before blocks take more rows
  s.threads = (int)std::min<int64_t>(1024, ((int64_t)s.rowsPerBlock * numTrees + 63) / 64 * 64);
  if (s.threads < 64) s.threads = 64;
  s.leafStride = (size_t)s.rowsPerBlock | 1; // (odd: the lanes that add a row's leaves read different banks)
  s.ldsBytes = ((size_t)numTrees * s.leafStride + (size_t)s.rowsPerBlock * numFeatures) * sizeof(float);
  s.ldsBytes = ((s.ldsBytes + 7) & ~(size_t)7) + (size_t)s.rowsPerBlock * std::max(1, numClasses) * sizeof(double);
  return s;
}

// The most rows of such a forest LaunchFewRows is used for (0: none).
constexpr int64_t kFewRowsWork = (int64_t)3 << 20; // (row, tree, block of three levels) visits
inline int64_t FewRowsMost(int32_t numFeatures, int32_t numTrees, int32_t numClasses, int32_t depth) {
  if (numTrees < 1) return 0;
  int64_t rows = kFewRowsWork / ((int64_t)numTrees * (depth / 3 + 1));
  while (rows > 0 && ShapeOfFewRows(rows, numFeatures, numTrees, numClasses).ldsBytes > kFewRowsLds) rows /= 2;
  return rows;
}

// How many rows of such a forest LaunchFewRows takes sooner than the launch plans do (0: never).  Two costs grow with the
// rows: the walks, about 20 cycles of a compute unit's address path per 16-byte gather of 64 lanes (4.5 us at kFewRowsWork
// visits), and the sums, 0.4 us per (row, class) that a wave adds.  A forest of many trees ends at the first, one of few
// trees (few waves a block) or many classes at the second.  Against it stand 7 us for the plans' launch and staging, 1.1 a
// class and up to 4 for the walk: fitted to 72 forests of 1 to 400 trees and 0 to 12 classes, 250 to 400000 rows each.
// Without the second term 393216 rows of two trees and two classes took 94 us here and 17 by the plan, 87381 rows of twelve
// trees and six classes 68 and 14; with it no forest of the fit is more than 1.3 times the faster of the two forms.
inline int64_t FewRowsLimit(int32_t numFeatures, int32_t numTrees, int32_t numClasses, int32_t depth) {
  const int64_t visits = (int64_t)numTrees * (depth / 3 + 1);
  const double planMicros = 7.0 + 1.1 * numClasses + std::min(4.0, (double)numTrees * depth / 100.0);
  int64_t rows = FewRowsMost(numFeatures, numTrees, numClasses, depth);
  for (; rows > 0; rows = rows * 7 / 8) {
    const FewRowsShape s = ShapeOfFewRows(rows, numFeatures, numTrees, numClasses);
    const int64_t waves = s.threads / 64, sums = ((int64_t)s.rowsPerBlock * std::max(1, numClasses) + waves - 1) / waves;
    if (4.5 + 4.5 * (double)(rows * visits) / (double)kFewRowsWork + 0.4 * (double)sums <= planMicros) break;
  }
  return rows;
}

// Rank-quantised rows (the output of LaunchBinRows) against bundles each wave streams on its own.
struct RankStreamParams {
  const uint8_t *ranks = nullptr;
  const uint32_t *words = nullptr; // PackRankStream
  const float *values = nullptr;
  const uint32_t *bundles = nullptr; // first words
  int64_t rows = 0;
  int32_t numFeatures = 0, numBundles = 0;
  int32_t chains = kStreamMaxChains;
  int32_t slices = 1;              // blocks that share a row block's bundles
  int32_t computeUnits = 256;
  int32_t transform = 0;
  double initialValue = 0.0;
  float *out = nullptr;            // one slice
  double *partial = nullptr;       // [slices][rows] otherwise
  hipEvent_t done = nullptr;
};

// Waves of a block of LaunchRankStream: as many as have room for two bundles each beside the rows' ranks.
constexpr int kStreamMaxWaves = 16;
constexpr int kStreamTilePieces = 6; // 16-byte pieces of the next rows' ranks that a lane holds in registers
inline int StreamWaves(int32_t numFeatures) {
  const int64_t tile = ((int64_t)(numFeatures + 1) * kStreamRows + 15) & ~(int64_t)15;
  return (int)std::min<int64_t>(kStreamMaxWaves, (160 * 1024 - tile) / (2 * kStreamBundleBytes));
}
// Slices fill the compute units while every wave of a block still has two bundles to overlap.
inline int32_t RankStreamSlices(int64_t rows, int32_t numFeatures, int32_t numBundles, int32_t computeUnits) {
  const int64_t blocks = (rows + kStreamRows - 1) / kStreamRows;
  const int64_t most = numBundles / (2 * std::max(1, StreamWaves(numFeatures)));
  return (int32_t)std::max<int64_t>(1, std::min<int64_t>({computeUnits / std::max<int64_t>(1, blocks), most, 64}));
}

// (Every launcher below records the `done` of its parameters behind its kernel.)
hipError_t LaunchFewRows(const FewRowsParams &p, hipStream_t stream);
hipError_t LaunchRankStream(const RankStreamParams &p, hipStream_t stream);

// Row-parallel walk over LDS-staged tree groups: block = s.rowsPerBlock * s.treeThreads lanes.
// `interleave` in {1,2,4,8}; `tileMode`: 0 f32 tile with byte offsets, 1 f32 tile with offsets in units of
// 4 bytes, 2 one-byte rank tile (p.x then points at the output of LaunchBinRows; 64 rows per block), 3 two-byte
// rank tile (p.x points at the output of LaunchRankRows16 for the same rowsPerBlock).
hipError_t LaunchWalkRowsLds(const WalkParams &p, int interleave, int tileMode, size_t ldsBytes, hipStream_t stream);
// The same block shape over tiled trees (tiles of 2 to 8 nodes, f32 row tile with byte offsets below 64 KB);
// `interleave` in {1,2,4}.  Tree groups are staged by direct global-to-LDS copies.
hipError_t LaunchWalkRowsTiled(const WalkParams &p, int tileSize, int interleave, size_t ldsBytes, hipStream_t stream);
// Rank-quantises rows x[rows][numFeatures] into ranks[ceil(rows/64)][numFeatures][64] (bytes) with the
// packer's threshold table ([chunk][k][64], +inf padded, tableDepth = 2^n - 1).
hipError_t LaunchBinRows(const float *x, const float *table, uint8_t *ranks, int64_t rows, int numFeatures,
                         int tableDepth, int chunkFeatures, hipStream_t stream);
// Ranks rows x[rows][numFeatures] into two-byte ranks laid out as [ceil(rows / rowsPerBlock)][(numFeatures + 2) / 2]
// [rowsPerBlock][2] with the packer's tables (PackedModel::rankTables / rankFeatures / rankChunks on the device);
// maxChunkEntries / maxChunkFeatures = the largest chunk's table entries / slots (the kernel's LDS need).  The rank
// buffer must hold the rows rounded up to whole row blocks and then to a multiple of 1024 rows.
hipError_t LaunchRankRows16(const float *x, const float *tables, const RankFeatureDesc *features, const RankChunkDesc *chunks,
                            int numChunks, uint32_t maxChunkEntries, uint32_t maxChunkFeatures, uint16_t *ranks, int64_t rows,
                            int numFeatures, int rowsPerBlock, hipStream_t stream);
// Tree-parallel walk: s.rowsPerBlock rows per block (row-major in LDS),
// s.treeLanes lanes per row; block = rowsPerBlock * treeLanes lanes.
hipError_t LaunchWalkTreeParallel(const WalkParams &p, int interleave, size_t ldsBytes, hipStream_t stream);
// Global-memory walk (fallback for trees that do not fit an LDS group): block = s.rowsPerBlock lanes,
// one per row; p.globalNodes / p.globalTrees instead of groups and bundles.
hipError_t LaunchWalkGlobal(const WalkParams &p, int interleave, hipStream_t stream);
hipError_t LaunchFinalize(const FinalizeParams &p, hipStream_t stream);

} // namespace tbamd
