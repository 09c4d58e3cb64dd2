// Device-facing model layout shared by the packer (host) and the HIP kernels.
//
// This replaces the reference's tiled-tree model buffers
// (src/utils/TreeTilingUtils.cpp:363-413 tile byte layout, :434-495
// offsets/lengths/classIds, src/mlir/Representations.cpp:1038-1052/:1728-1744
// tile structs, src/gpu/GPURepresentations.cpp:90-256 device packing) with a
// layout made for staging whole tree groups in LDS:
//
//  * A forest is cut into GROUPS of trees; one group's nodes are a contiguous
//    run of 8-byte nodes that is copied verbatim into LDS, so every pointer a
//    node holds is a byte address relative to the start of its group.
//  * Node = { f32 value; u32 meta }.  value is the split threshold or, on a
//    leaf, the prediction.  meta = (feature offset << 16) | left-child byte
//    address (that way round: a 16-bit addition to the low half is cheaper on
//    the device than one that selects the high half).  The right child always
//    follows the left one (+8 bytes).
//  * The feature offset is pre-multiplied for the transposed row tile the
//    kernel keeps in LDS (feature-major, one column per row of the block), so
//    the address of the feature value is `featureOffset + 4*rowSlot`.
//  * A leaf points at itself and tests the pad feature (index numFeatures),
//    whose column holds -inf: `x < value` is then always true, the walk takes
//    the "left" pointer and stays on the leaf.  A walk of `depth` steps thus
//    needs no leaf test: it ends on the leaf for every row.
//  * Leaves outside (PackedModel::leavesOutside): a walk's last step needs no node of the level it leads to, only which leaf it
//    is.  The leaves on the last level of a bundle's walk can therefore stay in global memory: behind the nodes that are copied
//    into LDS the group's image holds their values, 4 bytes each, siblings side by side (the last step adds 4 bytes for the right
//    one), and the walk ends with one read of the image at the address it arrived at, wherever that leaf stands.
//  * Deferred tails (LaunchPlan::deferTails; the reference's peeled walks for skewed trees,
//    src/mlir/ProbabilityBasedTilingTransform.cpp:66-73, src/mlir/WalkDecisionTreeLoweringPass.cpp:231-315): the
//    lock-step walk of a tree may stop at a level above its leaves.  The internal nodes of that level are then
//    represented by STUBS, which hold the walk in place like a leaf: the value field is a NaN (every compare
//    fails, the walk takes the "right" child) and the child pointer is the stub's own address minus one node, so
//    the right child is the stub itself.  The NaN's payload is the index of the node the stub stands for in the
//    TAIL ARRAY: the subtrees below the stubs stay in global memory, out of the tree groups, as nodes
//    { value; (left child index << kTailFeatureBits) | feature index } (PackedModel::tailNodes).  A model with a
//    NaN leaf value keeps its trees whole.
//  * Trees are walked K at a time (a BUNDLE) to give every lane K independent
//    dependency chains.  A bundle records the K root addresses, the trip count
//    (deepest tree of the bundle) and the class the trees add to.
//
// Tiled layout (LaunchPlan::tileSize T in 2..8; the reference's tile of T connected internal nodes,
// src/mlir/UniformTilingTransformation.cpp:148-195, src/mlir/ProbabilityBasedTilingTransform.cpp:124-198):
//  * A TILE holds its nodes in level order, struct-of-arrays: T thresholds, T feature offsets, the byte
//    address of its first child tile and a child-select table, in 16 / 24 / 32 bytes for T = 2 / 3 / 4:
//      T = 2: { f32 thr[2]; u16 off[2]; u16 childBase; u16 select }                      one 16-byte read
//      T = 3: { f32 thr[3]; u16 off[3]; u16 childBase; u16 select; u16 pad }             three 8-byte reads
//      T = 4: { f32 thr[4]; u16 off[4]; u16 childBase; u16 selectLow; u32 selectHigh }   two 16-byte reads
//  * The children of a tile (tiles or leaves, numbered left to right as in
//    docs/TileShapesAndLUT/TileShapesAndLUT.md:23-27) are consecutive tiles, child c at childBase + c * tile
//    bytes.  `select` is the tile's own row of the reference's LUT[shape][outcome]
//    (src/utils/TreeTilingUtils.cpp:1932-2018): field number `outcome` (2 bits wide for T <= 3, 3 bits for
//    T = 4) is the child reached when bit i of `outcome` says that node i's predicate held (node 0 in the
//    least significant bit, src/mlir/CodeGenStateMachine.cpp:284-506).  Keeping the row in the tile saves the
//    shape id and the table lookup.
//  * Unused node slots of a short tile test the pad feature; their outcome bits are don't-cares of `select`.
//  * A leaf is a tile of its own: thr[0] is the prediction, every slot tests the pad feature, childBase is
//    the tile's own address and select is 0, so a walk of `depth` tile steps needs no leaf test either.
//  * Tile sizes 5 to 8 share one 64-byte tile of eight slots (four 16-byte reads), the reference's default
//    tile size 8 among them (test/python/cpu_tests.py:14, src/test/GPUTests.cpp:995):
//      { f32 thr[8]; u16 off[8]; u64 links; u16 childBase; u16 pad[3] }
//    A table of 256 outcomes does not fit a tile, and one row of the reference's LUT per shape present in a
//    model (1430 shapes of 256 entries) fits no LDS, so the tile carries its own shape instead: `links` holds
//    a 4-bit link per slot and outcome, nibble s of the high word taken when slot s sends the row left (its
//    predicate holds) and nibble s of the low word when it sends it right.  A link below 7 names the next slot
//    (link + 1: slot 0 is nobody's child), a link of 7 or more the child reached (link - 7, children numbered
//    left to right, 0..8).  A tile step picks the eight links its comparisons select with one masked insert of
//    the high word into the low one and follows them from slot 0, as many as the tiles of the model have
//    levels of nodes; this is the reference's LUT[shape][outcome] evaluated instead of stored, so the outcome
//    bit order and the child numbering are the same.  A leaf tile's links
//    all say "child 0" and its childBase is its own address.
#pragma once

#include <cstdint>

namespace tbamd {

constexpr int kMaxInterleave = 8;
constexpr uint32_t kNodeBytes = 8;
constexpr uint32_t kDeferBytesPerWave = 512; // LDS of one wave's queue of deferred walks (LaunchPlan::deferTails)
// Deferred tails: a tail node's meta word holds the index of its left child above kTailFeatureBits bits of feature
// index; a queue entry holds a tail index below 6 bits of lane (bits 26 to 31).
// (Eight bits: a row tile with byte offsets holds 64 rows of at most 255 features and the pad feature.)
constexpr uint32_t kTailFeatureBits = 8;
constexpr uint32_t kMaxTailNodes = 1u << 22;
// A stub's value field: a quiet NaN whose low bits are the tail index.
constexpr uint32_t kStubValueBits = 0x7FC00000u;
constexpr uint32_t kStubIndexMask = kMaxTailNodes - 1u;
constexpr int kMaxTileSize = 8;
// Tiles of more than kMaxSelectTile nodes carry links instead of a child-select table.
constexpr int kMaxSelectTile = 4;
// Bytes of one tile of T nodes (T = 1 is the scalar node).
constexpr uint32_t TileBytes(int tileSize) {
  return tileSize <= 1 ? kNodeBytes : tileSize == 2 ? 16u : tileSize == 3 ? 24u : tileSize == 4 ? 32u : 64u;
}
// Width of one field of a tile's child-select table (tiles of up to kMaxSelectTile nodes).
constexpr uint32_t TileSelectBits(int tileSize) { return tileSize == 4 ? 3u : 2u; }
// Links of the 64-byte tile: values below kTileLinkExit name a slot (value + 1), the others a child (value - kTileLinkExit).
constexpr uint32_t kTileLinkExit = 7;
constexpr uint64_t kLeafTileLinks = 0x7777777777777777ull; // every link: child 0

struct DeviceNode {
  float value;
  uint32_t meta;
};
constexpr uint32_t NodeMeta(uint32_t child, uint32_t featureOffset) { return featureOffset << 16 | child; }
constexpr uint32_t MetaChild(uint32_t meta) { return meta & 0xFFFFu; }
constexpr uint32_t MetaFeature(uint32_t meta) { return meta >> 16; }

struct alignas(32) DeviceBundle {
  uint16_t root[kMaxInterleave]; // byte address of each tree's root inside the group
  uint32_t depth;                // walk steps (tile steps in the tiled layout) that bring every row to a leaf (or to a stub)
  // (Bit fields of one word, which a scalar load fetches: there is none of 16 bits, and a vector load in its place has a bundle wait
  // for memory, and for every leaf value on its way: 2^20 rows x 800 trees x 8 classes 727 -> 694 us.)
  uint32_t classId : 16;
  uint32_t hasStubs : 16;        // deferred tails: some tree of the bundle ends in stubs
  uint32_t firstSlot;            // index of root[0] in the slot->tree table
  uint32_t peelDepth;            // steps taken without looking; the rest runs while any lane still moves (== depth: no tail)
};

// Node of the global-memory walk (trees too big for an LDS group): 16 bytes, absolute indices.
struct DeviceGlobalNode {
  float value;        // threshold, or the prediction on a leaf
  uint32_t feature;   // feature index; kGlobalLeaf on a leaf
  uint32_t left;      // index of the left child in the node array (right = left + 1)
  int32_t origin;     // node id in the model file's numbering
};
constexpr uint32_t kGlobalLeaf = 0xFFFFFFFFu;

// Per-tree record of the global-memory walk.
struct DeviceGlobalTree {
  uint32_t root;
  uint32_t depth;
  uint32_t classId;
  int32_t origin;     // tree index in the model file
};

// Ranking kernel of the two-byte rank rows: where a feature's threshold table (a complete search tree in
// breadth-first order, 2^levels - 1 entries) starts inside its chunk, and which whole feature pairs a chunk holds.
struct RankFeatureDesc {
  uint32_t tableOffset;
  uint32_t levels;
};
struct RankChunkDesc {
  uint32_t firstFeature, numFeatures;
  uint32_t tableBegin, tableEntries;
};

// Three levels of a tree in one 48-byte piece (three 16-byte loads), for walks whose cost is the latency of dependent
// loads: slot 0 is the top node, slots 1-2 its children, slots 3-6 theirs, the eight children below those are the
// tops of further blocks.  A leaf (feature kFewRowsLeaf) ends the walk in whatever slot it sits; the children of
// slots 3-6 that exist (bit 2 * (slot - 3) + side of `exits`) follow each other from block `firstChild`.
struct DeviceFewRowsBlock {
  float value[7];       // split threshold, or the prediction on a leaf
  uint32_t firstChild;
  uint16_t feature[7];
  uint16_t exits;
};
static_assert(sizeof(DeviceFewRowsBlock) == 48, "three 16-byte loads");
constexpr uint32_t kFewRowsLeaf = 0xFFFFu;

// Rank-quantised rows of up to 2047 features, trees of up to 255 splits: 4-byte nodes that a wave streams through LDS of
// its own.  node = test << 24 | child pair << 16 | feature << 5: a row whose rank is below `test` (threshold index + 1)
// goes to word 2 * pair of the tree, the others to word 2 * pair + 1; word 0 is the root, word 1 unused: the bundle's head
// holds the root, and only a tree that is one leaf has the two.  A leaf holds
// its place: as a left child it tests the pad feature (rank 0) against 1, as a right child anything against 0.  The
// leaves a walk of the bundle's depth reaches with its last step are never read as nodes: they have no words.
// Predictions stand in an array of their own, one place per word (the last leaves' included).
//
// A bundle's image begins with a DeviceStreamHead for each half of the wave that walks it, then the trees; it starts on a
// 16-byte piece and the copy takes kStreamBundleBytes whatever its size (the words end with as many that belong to none).
struct alignas(16) DeviceStreamHead {
  uint16_t roots[4];      // byte offsets of the half's trees in the image (of their word 0, which may lie in front of their words)
  uint32_t depth;         // of the deepest tree of the bundle, at least 1
  uint32_t words;         // of the image (what reads it on the host checks against)
  uint32_t rootWords[4];  // word 0 of every tree
  uint32_t valueBegin[4]; // of every tree, in the array of predictions (entry 0 is 0.0: the empty places')
};
static_assert(sizeof(DeviceStreamHead) == 48, "three 16-byte LDS reads");
constexpr uint32_t kStreamHeadWords = 2 * sizeof(DeviceStreamHead) / 4;
constexpr int kStreamMaxChains = 4;          // trees a lane walks side by side (2 or 4); two lanes share a bundle's trees
constexpr uint32_t kStreamBundleBytes = 4096;
constexpr int32_t kStreamMaxFeatures = 2047;
constexpr int32_t kStreamRows = 32;          // rows of a block: a rank byte each, 32 per feature

struct DeviceGroup {
  uint32_t nodeBegin;   // first node of the group in the packed node array
  uint32_t nodeCount;   // multiple of 2 so that the group is a whole number of 16-byte pieces
  uint32_t bundleBegin;
  uint32_t bundleCount;
  uint32_t uniformClass; // class id + 1 when every bundle of the group votes for one class, else 0
  uint32_t imageCount;   // 8-byte units of the group's image: nodeCount of them in LDS, behind them the leaves that are not, 4 bytes each
  uint32_t reserved[2];
};
static_assert(sizeof(DeviceGroup) == 32, "group descriptors are fetched with one 32-byte scalar load");

} // namespace tbamd
