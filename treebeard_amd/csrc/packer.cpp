#include "packer.h"

#include <algorithm>
#include <cmath>
#include <functional>
#include <limits>
#include <cstring>
#include <numeric>

namespace tbamd {

Forest NormalizeToLessThan(const Forest &forest) {
  if (forest.predicate == Predicate::kLT) return forest;
  Forest out = forest;
  out.predicate = Predicate::kLT;
  const bool swapChildren = forest.predicate == Predicate::kGE || forest.predicate == Predicate::kGT;
  // x <= t  <=>  x < nextafter(t, +inf)   and   x > t  <=>  !(x <= t)
  const bool bumpThreshold = forest.predicate == Predicate::kLE || forest.predicate == Predicate::kGT;
  for (auto &tree : out.trees)
    for (size_t i = 0; i < tree.NumNodes(); ++i) {
      if (tree.IsLeaf((int32_t)i)) continue;
      if (bumpThreshold) tree.value[i] = std::nextafter(tree.value[i], std::numeric_limits<float>::infinity());
      if (swapChildren) std::swap(tree.left[i], tree.right[i]);
    }
  return out;
}

uint32_t PackedModel::PadFeatureOffset() const { return plan.FeatureOffset((uint32_t)numFeatures); }

size_t PackedModel::RowTileBytes() const {
  if (plan.rankRows16) return (size_t)((numFeatures + 2) / 2) * plan.rowsPerBlock * 4; // pairs of two-byte ranks, pad feature included
  return (size_t)(numFeatures + 1) * plan.rowsPerBlock * (plan.quantizedRows ? 1 : 4); // (+ the pad feature's column)
}

size_t PackedModel::LdsBytes() const {
  if (plan.kernel == LaunchPlan::Kernel::kGlobalWalk) return 0;
  size_t bytes = RowTileBytes() + (size_t)GroupRegionBytes();
  if (plan.kernel == LaunchPlan::Kernel::kTreeParallel) {
    // cross-wave reduction scratch + per-row, per-class accumulators (doubles)
    const size_t waves = (size_t)(plan.ThreadsPerBlock() + 63) / 64;
    bytes = (bytes + 7) & ~(size_t)7;
    bytes += waves * 8 + (size_t)plan.rowsPerBlock * (numClasses > 0 ? numClasses : 1) * 8;
  } else if (plan.treeThreads > 1 && numClasses > 0 && !ownClasses) {
    bytes = (bytes + 7) & ~(size_t)7;
    bytes += (size_t)plan.ThreadsPerBlock() * 8; // classifiers: cross-wave pass behind the row tile
  }
  if (plan.deferTails) {
    bytes = (bytes + 15) & ~(size_t)15;
    bytes += (size_t)(plan.ThreadsPerBlock() / 64) * kDeferBytesPerWave; // every wave's queue of deferred walks
  }
  return bytes;
}

namespace {

// Sorted distinct thresholds per feature of a forest already normalised to "x < t".
std::vector<std::vector<float>> ThresholdsPerFeature(const Forest &forest) {
  std::vector<std::vector<float>> out((size_t)forest.numFeatures);
  for (auto &tree : forest.trees) { // (of the splits that walks reach: nothing is known of others)
    std::vector<int32_t> stack{0};
    while (!stack.empty()) {
      const int32_t n = stack.back();
      stack.pop_back();
      if (tree.IsLeaf(n)) continue;
      out[(size_t)tree.feature[n]].push_back(tree.value[n]);
      stack.push_back(tree.left[n]);
      stack.push_back(tree.right[n]);
    }
  }
  for (auto &v : out) {
    std::sort(v.begin(), v.end());
    v.erase(std::unique(v.begin(), v.end()), v.end());
  }
  return out;
}

} // namespace

int32_t MaxThresholdsPerFeature(const Forest &forest) {
  size_t most = 0;
  for (auto &v : ThresholdsPerFeature(NormalizeToLessThan(forest))) most = std::max(most, v.size());
  return (int32_t)most;
}

namespace {

// Level-order node list of one tree with siblings adjacent.
struct LevelOrder {
  std::vector<int32_t> order;    // packed position -> original node
  std::vector<int32_t> position; // original node -> packed position
};

LevelOrder MakeLevelOrder(const Tree &tree) {
  LevelOrder lo;
  lo.position.assign(tree.NumNodes(), -1);
  lo.order.push_back(0);
  for (size_t head = 0; head < lo.order.size(); ++head) {
    int32_t n = lo.order[head];
    lo.position[n] = (int32_t)head;
    if (tree.IsLeaf(n)) continue;
    lo.order.push_back(tree.left[n]);
    lo.order.push_back(tree.right[n]);
  }
  return lo;
}

} // namespace


namespace {

// ---------------------------------------------------------------------------
// Tiling of one tree (LaunchPlan::tileSize > 1).
// ---------------------------------------------------------------------------
struct TileInfo {
  int32_t count = 0;                       // internal nodes in the tile; 0: a leaf tile
  int32_t members[kMaxTileSize] = {};      // original node ids, level order inside the tile
  int32_t numExits = 0;
  int32_t exits[kMaxTileSize + 1] = {};    // original node ids the tile's children start at, left to right
  int32_t leafNode = -1;                   // leaf tiles: the original leaf
  uint32_t firstChild = 0;                 // tile index (inside the tree) of child 0; own index on a leaf tile
  uint64_t select = 0;                     // child number per outcome word, TileSelectBits() each (tiles of up to 4 nodes)
  uint64_t links = kLeafTileLinks;         // a 4-bit link per slot and outcome (tiles of 5 to 8 nodes, device_model.h)
  int32_t hops = 1;                        // links a walk follows inside the tile at most (its levels of nodes)
  int32_t depth = 0;                       // tile steps from this tile down to its deepest leaf
  int32_t level = 0;                       // tile steps from the root tile
};

struct TiledTree {
  std::vector<TileInfo> tiles; // children of a tile are consecutive
  int32_t depth = 0;           // tile steps that bring every row to a leaf tile
  int32_t hops = 1;            // the most levels of nodes any tile holds
  bool byProfile = false;
};

// Members of the tile rooted at `root`, breadth first over internal nodes, left before right
// (src/mlir/UniformTilingTransformation.cpp:148-168).
int GatherUniform(const Tree &tree, int32_t root, int T, int32_t *members) {
  int32_t queue[2 * kMaxTileSize + 2];
  int head = 0, tail = 0, n = 0;
  queue[tail++] = root;
  while (head < tail && n < T) {
    const int32_t node = queue[head++];
    members[n++] = node;
    if (!tree.IsLeaf(tree.left[node])) queue[tail++] = tree.left[node];
    if (!tree.IsLeaf(tree.right[node])) queue[tail++] = tree.right[node];
  }
  return n;
}

// Members chosen by visit counts: the tile grows by the most-visited internal child of any member
// (src/mlir/ProbabilityBasedTilingTransform.cpp:152-190: members are scanned in node order, left child before
// right, and a candidate wins only with strictly more hits).
int GatherByHits(const Tree &tree, const std::vector<int64_t> &hits, int32_t root, int T, int32_t *members) {
  int n = 0;
  members[n++] = root;
  while (n < T) {
    int32_t sorted[kMaxTileSize];
    std::copy(members, members + n, sorted);
    std::sort(sorted, sorted + n);
    int64_t bestHits = -1;
    int32_t best = -1;
    for (int i = 0; i < n; ++i)
      for (int32_t child : {tree.left[sorted[i]], tree.right[sorted[i]]}) {
        if (tree.IsLeaf(child) || hits[child] <= bestHits) continue;
        if (std::find(members, members + n, child) != members + n) continue;
        bestHits = hits[child];
        best = child;
      }
    if (best < 0) break;
    members[n++] = best;
  }
  return n;
}

// src/mlir/ProbabilityBasedTilingTransform.cpp:208-225: the most-visited tenth of the leaves takes more
// than 90 % of the rows.
bool IsSkewed(const Tree &tree, const std::vector<int64_t> &hits) {
  std::vector<int64_t> leafHits;
  for (size_t i = 0; i < tree.NumNodes(); ++i)
    if (tree.IsLeaf((int32_t)i)) leafHits.push_back(hits[i]);
  std::sort(leafHits.begin(), leafHits.end(), std::greater<int64_t>());
  const size_t consider = (size_t)((double)leafHits.size() * 0.10);
  int64_t covered = 0;
  for (size_t i = 0; i < consider; ++i) covered += leafHits[i];
  return hits[0] > 0 && (double)covered / (double)hits[0] > 0.9;
}

TiledTree TileTree(const Tree &tree, int T, int tiling, const std::vector<int64_t> *hits) {
  TiledTree out;
  out.byProfile = tiling != 0 && hits != nullptr && IsSkewed(tree, *hits);
  // depth of every original node, for the level order inside a tile
  std::vector<int32_t> nodeDepth(tree.NumNodes(), -1);
  {
    std::vector<int32_t> stack{0};
    nodeDepth[0] = 0;
    while (!stack.empty()) {
      const int32_t n = stack.back();
      stack.pop_back();
      if (tree.IsLeaf(n)) continue;
      nodeDepth[tree.left[n]] = nodeDepth[tree.right[n]] = nodeDepth[n] + 1;
      stack.push_back(tree.left[n]);
      stack.push_back(tree.right[n]);
    }
  }
  std::vector<int32_t> roots{0}; // node each tile starts at, in tile order
  for (size_t ti = 0; ti < roots.size(); ++ti) {
    TileInfo tile;
    const int32_t root = roots[ti];
    if (tree.IsLeaf(root)) {
      tile.leafNode = root;
      tile.firstChild = (uint32_t)ti;
      out.tiles.push_back(tile);
      continue;
    }
    bool byHits = out.byProfile;
    if (byHits && tiling == 2 && (double)(*hits)[root] / (double)(*hits)[0] < 0.20) byHits = false; // hybrid
    int32_t members[kMaxTileSize];
    const int n = byHits ? GatherByHits(tree, *hits, root, T, members) : GatherUniform(tree, root, T, members);
    // level order inside the tile: by depth, then left to right (position in an in-order walk of the tile)
    std::vector<int32_t> inorder;
    {
      // in-order walk restricted to the members
      std::vector<std::pair<int32_t, int>> stack{{root, 0}};
      while (!stack.empty()) {
        auto [node, state] = stack.back();
        stack.pop_back();
        const bool member = std::find(members, members + n, node) != members + n;
        if (!member) continue;
        if (state == 0) {
          stack.push_back({node, 1});
          stack.push_back({tree.left[node], 0});
        } else {
          inorder.push_back(node);
          stack.push_back({tree.right[node], 0});
        }
      }
    }
    std::vector<int32_t> ordered(members, members + n);
    std::stable_sort(ordered.begin(), ordered.end(), [&](int32_t a, int32_t b) {
      if (nodeDepth[a] != nodeDepth[b]) return nodeDepth[a] < nodeDepth[b];
      return std::find(inorder.begin(), inorder.end(), a) < std::find(inorder.begin(), inorder.end(), b);
    });
    tile.count = n;
    std::copy(ordered.begin(), ordered.end(), tile.members);
    // tile-local children (slot or -(exit number) - 1), exits numbered left to right
    int32_t leftSlot[kMaxTileSize], rightSlot[kMaxTileSize];
    auto slotOf = [&](int32_t node) {
      for (int i = 0; i < n; ++i)
        if (tile.members[i] == node) return i;
      return -1;
    };
    {
      std::vector<std::pair<int, int>> stack{{0, 0}};
      while (!stack.empty()) {
        auto [slot, state] = stack.back();
        stack.pop_back();
        const int32_t node = tile.members[slot];
        if (state == 0) {
          stack.push_back({slot, 1});
          const int child = slotOf(tree.left[node]);
          if (child >= 0) {
            leftSlot[slot] = child;
            stack.push_back({child, 0});
          } else {
            leftSlot[slot] = -(tile.numExits) - 1;
            tile.exits[tile.numExits++] = tree.left[node];
          }
        } else {
          const int child = slotOf(tree.right[node]);
          if (child >= 0) {
            rightSlot[slot] = child;
            stack.push_back({child, 0});
          } else {
            rightSlot[slot] = -(tile.numExits) - 1;
            tile.exits[tile.numExits++] = tree.right[node];
          }
        }
      }
    }
    if (T <= kMaxSelectTile) {
      // the tile's row of the child look-up table: outcome bit i set = node i sends the row left
      const uint32_t width = TileSelectBits(T);
      for (uint32_t outcome = 0; outcome < (1u << T); ++outcome) {
        int slot = 0;
        for (;;) {
          const int32_t next = ((outcome >> slot) & 1u) ? leftSlot[slot] : rightSlot[slot];
          if (next < 0) {
            tile.select |= (uint64_t)(-next - 1) << (outcome * width);
            break;
          }
          slot = next;
        }
      }
    } else {
      // the tile's shape itself: per slot where a row goes when the slot's predicate holds (left) and when not
      auto link = [](int32_t next) -> uint64_t { return next < 0 ? kTileLinkExit + (uint64_t)(-next - 1) : (uint64_t)(next - 1); };
      tile.links = 0;
      for (int slot = 0; slot < kMaxTileSize; ++slot) {
        const uint64_t left = slot < n ? link(leftSlot[slot]) : kTileLinkExit, right = slot < n ? link(rightSlot[slot]) : kTileLinkExit;
        tile.links |= (right << (4 * slot)) | (left << (32 + 4 * slot));
      }
      for (int i = 0; i < n; ++i) tile.hops = std::max(tile.hops, nodeDepth[tile.members[i]] - nodeDepth[tile.members[0]] + 1);
      out.hops = std::max(out.hops, tile.hops);
    }
    tile.firstChild = (uint32_t)roots.size();
    for (int e = 0; e < tile.numExits; ++e) roots.push_back(tile.exits[e]);
    out.tiles.push_back(tile);
  }
  // levels top down (children follow their parent in tile order), depths bottom up
  for (size_t ti = 0; ti < out.tiles.size(); ++ti)
    for (int e = 0; e < out.tiles[ti].numExits; ++e)
      out.tiles[out.tiles[ti].firstChild + e].level = out.tiles[ti].level + 1;
  for (size_t ti = out.tiles.size(); ti-- > 0;) {
    TileInfo &tile = out.tiles[ti];
    for (int e = 0; e < tile.numExits; ++e) tile.depth = std::max(tile.depth, 1 + out.tiles[tile.firstChild + e].depth);
  }
  out.depth = out.tiles[0].depth;
  return out;
}

// Bytes of one tile (see device_model.h) for a tree whose tile 0 sits at byte address `treeBase` of its group.
void EmitTile(const Tree &tree, const TileInfo &tile, int T, uint32_t treeBase, size_t tileIndex, uint32_t featureStride,
              uint32_t padOffset, unsigned char *dst) {
  const uint32_t bytes = TileBytes(T);
  float thr[kMaxTileSize] = {};
  uint16_t off[kMaxTileSize];
  for (int i = 0; i < kMaxTileSize; ++i) off[i] = (uint16_t)padOffset;
  if (tile.count == 0) {
    thr[0] = tree.value[tile.leafNode];
  } else {
    for (int i = 0; i < tile.count; ++i) {
      thr[i] = tree.value[tile.members[i]];
      off[i] = (uint16_t)((uint32_t)tree.feature[tile.members[i]] * featureStride);
    }
  }
  const uint32_t childAddress = treeBase + tile.firstChild * bytes;
  if (childAddress + (uint32_t)std::max(tile.numExits, 1) * bytes > 0x10000u) throw Error("internal error: tile address beyond the group");
  const uint16_t childBase = (uint16_t)childAddress;
  std::memset(dst, 0, bytes);
  if (T > kMaxSelectTile) { // eight slots whatever the tile size: { thr[8]; off[8]; links; childBase }
    std::memcpy(dst, thr, 32);
    std::memcpy(dst + 32, off, 16);
    std::memcpy(dst + 48, &tile.links, 8);
    std::memcpy(dst + 56, &childBase, 2);
    return;
  }
  std::memcpy(dst, thr, (size_t)T * 4);
  std::memcpy(dst + T * 4, off, (size_t)T * 2);
  std::memcpy(dst + T * 6, &childBase, 2);
  if (T == 4) {
    const uint16_t low = (uint16_t)(tile.select & 0xFFFFu);
    const uint32_t high = (uint32_t)(tile.select >> 16);
    std::memcpy(dst + 26, &low, 2);
    std::memcpy(dst + 28, &high, 4);
  } else {
    const uint16_t select = (uint16_t)tile.select;
    std::memcpy(dst + T * 6 + 2, &select, 2);
  }
  (void)tileIndex;
}

// Steps after which 90 % of the profiled rows of a tree have reached their leaf
// (src/utils/TreeTilingUtils.cpp:1722-1743); `leafLevel[i]` is the step count of leaf i, -1 for other nodes.
int32_t PeelDepth(const std::vector<int64_t> &hits, const std::vector<int32_t> &leafLevel, int32_t depth) {
  if (hits.empty() || hits[0] <= 0) return depth;
  for (int32_t d = 0; d <= depth; ++d) {
    int64_t covered = 0;
    for (size_t i = 0; i < leafLevel.size(); ++i)
      if (leafLevel[i] >= 0 && leafLevel[i] <= d) covered += hits[i];
    if ((double)covered / (double)hits[0] >= 0.9) return d;
  }
  return depth;
}

} // namespace

int64_t BiggestTiledTreeBytes(const Forest &forest, int tileSize) {
  if (tileSize < 2 || tileSize > kMaxTileSize) throw Error("internal error: tile size out of range");
  size_t most = 0;
  for (const Tree &tree : forest.trees) most = std::max(most, TileTree(tree, tileSize, 0, nullptr).tiles.size());
  return (int64_t)most * TileBytes(tileSize);
}

namespace {

// Global-memory layout: every tree breadth first (siblings adjacent), absolute node indices.
PackedModel PackForGlobalWalk(const Forest &forest, const LaunchPlan &plan) {
  if (plan.rowsPerBlock < 64 || plan.rowsPerBlock > 1024 || plan.rowsPerBlock % 64 != 0)
    throw Error("the global-memory walk needs a block of 64..1024 lanes");
  PackedModel pm;
  pm.plan = plan;
  pm.numFeatures = forest.numFeatures;
  pm.numClasses = forest.numClasses;
  pm.numTrees = (int32_t)forest.trees.size();
  std::vector<int32_t> depth(forest.trees.size());
  for (size_t t = 0; t < forest.trees.size(); ++t) depth[t] = forest.trees[t].Depth();
  std::vector<int32_t> order(forest.trees.size());
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
    const int32_t ca = forest.numClasses > 0 ? forest.trees[a].classId : 0;
    const int32_t cb = forest.numClasses > 0 ? forest.trees[b].classId : 0;
    if (ca != cb) return ca < cb;
    return depth[a] < depth[b];
  });
  if (forest.NumNodes() > 0x7FFFFFF0u) throw Error("forest has too many nodes");
  for (int32_t t : order) {
    const Tree &tree = forest.trees[t];
    const LevelOrder lo = MakeLevelOrder(tree);
    const uint32_t base = (uint32_t)pm.globalNodes.size();
    pm.globalTrees.push_back(DeviceGlobalTree{base, (uint32_t)depth[t],
                                              (uint32_t)(forest.numClasses > 0 ? tree.classId : 0), t});
    for (size_t i = 0; i < lo.order.size(); ++i) {
      const int32_t n = lo.order[i];
      DeviceGlobalNode dn;
      dn.value = tree.value[n];
      dn.origin = n;
      if (tree.IsLeaf(n)) {
        dn.feature = kGlobalLeaf;
        dn.left = base + (uint32_t)i;
      } else {
        dn.feature = (uint32_t)tree.feature[n];
        dn.left = base + (uint32_t)lo.position[tree.left[n]];
      }
      pm.globalNodes.push_back(dn);
    }
  }
  return pm;
}

} // namespace

RankStreamModel PackRankStream(const Forest &input) {
  RankStreamModel sm;
  if (input.numClasses > 0 || input.numFeatures > kStreamMaxFeatures || input.trees.empty()) return sm;
  const Forest forest = NormalizeToLessThan(input);
  const std::vector<std::vector<float>> ranks = ThresholdsPerFeature(forest);
  for (auto &sorted : ranks)
    if (sorted.size() > 254) return sm;
  std::vector<int32_t> order(forest.trees.size()), depth(forest.trees.size());
  for (size_t t = 0; t < forest.trees.size(); ++t) {
    if (forest.trees[t].NumNodes() > 511) return sm;
    depth[t] = forest.trees[t].Depth();
  }
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
    return depth[(size_t)a] != depth[(size_t)b] ? depth[(size_t)a] < depth[(size_t)b]
                                                : forest.trees[(size_t)a].NumNodes() < forest.trees[(size_t)b].NumNodes();
  });
  auto leafWord = [&](uint32_t pair, bool right) { return (right ? 0u : 1u << 24) | pair << 16 | (uint32_t)forest.numFeatures << 5; };
  // words of a tree's image in a bundle of `deepest` levels: the children of level deepest - 1 have none, nor has a root that splits
  auto wordsOf = [&](int32_t t, int32_t deepest) {
    const Tree &tree = forest.trees[(size_t)t];
    std::vector<int32_t> level{0};
    uint32_t words = 2;
    for (int32_t d = 0; d + 1 < deepest && !level.empty(); ++d) {
      std::vector<int32_t> below;
      for (int32_t n : level)
        if (!tree.IsLeaf(n)) below.insert(below.end(), {tree.left[(size_t)n], tree.right[(size_t)n]});
      words += (uint32_t)below.size();
      level.swap(below);
    }
    return tree.IsLeaf(0) ? words : words - 2;
  };
  auto pack = [&](int32_t chains) {
    sm = RankStreamModel();
    sm.chains = chains;
    sm.values.push_back(0.0f);
    for (size_t next = 0; next < order.size();) {
      // as many trees as fit, each with the words the deepest of them (the last: they come by depth) asks for
      size_t count = 0;
      for (size_t n = 1; n <= (size_t)(2 * chains) && next + n <= order.size(); ++n) {
        uint32_t words = kStreamHeadWords + 2 + 3;
        for (size_t k = 0; k < n; ++k) words += wordsOf(order[next + k], depth[(size_t)order[next + n - 1]]);
        if (words * 4 > kStreamBundleBytes && n > 1) break; // (a tree alone always fits)
        count = n;
      }
      const int32_t deepest = std::max(1, depth[(size_t)order[next + count - 1]]);
      const uint32_t begin = (uint32_t)sm.words.size();
      DeviceStreamHead heads[2]{};
      for (DeviceStreamHead &head : heads) {
        for (uint16_t &root : head.roots) root = kStreamHeadWords * 4; // (the empty tree)
        for (uint32_t &word : head.rootWords) word = leafWord(0, false);
        head.depth = (uint32_t)deepest;
      }
      sm.words.resize(begin + kStreamHeadWords);
      sm.words.insert(sm.words.end(), {leafWord(0, false), 0u}); // the empty tree
      for (size_t k = 0; k < count; ++k) {
        const int32_t t = order[next + k];
        const Tree &tree = forest.trees[(size_t)t];
        const uint32_t own = wordsOf(t, deepest), inHead = tree.IsLeaf(0) ? 0u : 2u, limit = own + inHead;
        const size_t at = sm.words.size() - inHead, valueAt = sm.values.size(); // (words 0 and 1 of a root that splits: the head's)
        heads[k & 1].roots[k / 2] = (uint16_t)((at - begin) * 4);
        heads[k & 1].valueBegin[k / 2] = (uint32_t)valueAt;
        sm.words.resize(sm.words.size() + own, 0u);
        sm.values.resize(valueAt + tree.NumNodes() + 1, 0.0f);
        struct Place { int32_t node; uint32_t word; };
        std::vector<Place> queue{{0, 0}};
        uint32_t pairs = 1;
        for (size_t head = 0; head < queue.size(); ++head) { // breadth first: the last level's words come last
          const auto [n, word] = queue[head];
          if (tree.IsLeaf(n)) {
            if (word < limit) sm.words[at + word] = leafWord(word / 2, word & 1u);
            if (word == 0) heads[k & 1].rootWords[k / 2] = leafWord(0, false);
            sm.values[valueAt + word] = tree.value[(size_t)n];
            continue;
          }
          const auto &sorted = ranks[(size_t)tree.feature[(size_t)n]];
          const uint32_t test = (uint32_t)(std::lower_bound(sorted.begin(), sorted.end(), tree.value[(size_t)n]) - sorted.begin()) + 1;
          if (word >= limit) throw Error("internal error: a split without a word");
          (word == 0 ? heads[k & 1].rootWords[k / 2] : sm.words[at + word]) =
              test << 24 | pairs << 16 | (uint32_t)tree.feature[(size_t)n] << 5;
          queue.push_back({tree.left[(size_t)n], 2 * pairs});
          queue.push_back({tree.right[(size_t)n], 2 * pairs + 1});
          ++pairs;
        }
      }
      while (sm.words.size() % 4) sm.words.push_back(0u);
      for (DeviceStreamHead &head : heads) head.words = (uint32_t)sm.words.size() - begin;
      std::memcpy(sm.words.data() + begin, heads, sizeof(heads));
      if (sm.words.size() > 0x7FFFFFF0u) throw Error("forest has too many nodes");
      sm.bundles.push_back(begin);
      next += count;
    }
    sm.words.resize(sm.words.size() + kStreamBundleBytes / 4, 0u);
  };
  // four chains where bundles of eight trees are mostly full: a chain of empty places costs what any other does
  pack(kStreamMaxChains);
  if (sm.bundles.size() * 6 > order.size() + 6) pack(2);
  return sm;
}

FewRowsModel PackFewRows(const Forest &input) {
  FewRowsModel fm;
  if (input.numFeatures >= (int32_t)kFewRowsLeaf) return fm;
  const Forest forest = NormalizeToLessThan(input);
  const int32_t Cn = std::max(1, forest.numClasses);
  std::vector<int32_t> order(forest.trees.size());
  std::iota(order.begin(), order.end(), 0);
  auto classOf = [&](int32_t t) { return forest.numClasses > 0 ? forest.trees[(size_t)t].classId : 0; };
  std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) { return classOf(a) < classOf(b); });
  fm.classBegin.assign((size_t)Cn + 1, (int32_t)order.size());
  for (size_t i = order.size(); i-- > 0;)
    for (int32_t c = classOf(order[i]); c >= 0 && fm.classBegin[(size_t)c] > (int32_t)i; --c) fm.classBegin[(size_t)c] = (int32_t)i;
  fm.blocks.resize(order.size());
  struct Top { int32_t node; size_t block; };
  std::vector<Top> queue;
  for (size_t i = 0; i < order.size(); ++i) {
    const Tree &tree = forest.trees[(size_t)order[i]];
    queue.assign(1, Top{0, i});
    for (size_t head = 0; head < queue.size(); ++head) {
      DeviceFewRowsBlock b{};
      for (uint16_t &f : b.feature) f = (uint16_t)kFewRowsLeaf; // (slots below a leaf are never reached)
      b.firstChild = (uint32_t)fm.blocks.size();
      int32_t at[7] = {queue[head].node, -1, -1, -1, -1, -1, -1};
      for (int s = 0; s < 7; ++s) {
        if (at[s] < 0) continue;
        const int32_t n = at[s];
        b.value[s] = tree.value[(size_t)n];
        if (tree.IsLeaf(n)) continue;
        b.feature[s] = (uint16_t)tree.feature[(size_t)n];
        for (int side = 0; side < 2; ++side) {
          const int32_t child = side == 0 ? tree.left[(size_t)n] : tree.right[(size_t)n];
          if (s < 3) {
            at[2 * s + 1 + side] = child;
          } else {
            b.exits = (uint16_t)(b.exits | 1u << (2 * (s - 3) + side));
            queue.push_back(Top{child, fm.blocks.size()});
            fm.blocks.emplace_back();
          }
        }
      }
      fm.blocks[queue[head].block] = b;
      if (fm.blocks.size() > 0x7FFFFFF0u) throw Error("forest has too many nodes");
    }
  }
  return fm;
}

namespace {
// A tree in a group's image, in units of 8 bytes.
struct TreeUnits {
  uint32_t whole = 0;
  uint32_t lowest = 0; // of which the leaves of its last level, where the walk can take those from global memory
};

// How many nodes that walks reach a tree has on each level.
std::vector<uint32_t> NodesPerLevel(const Tree &tree) {
  std::vector<uint32_t> counts;
  std::vector<int32_t> level{0}, below;
  while (!level.empty()) {
    counts.push_back((uint32_t)level.size());
    below.clear();
    for (int32_t n : level)
      if (!tree.IsLeaf(n)) below.insert(below.end(), {tree.left[(size_t)n], tree.right[(size_t)n]});
    level.swap(below);
  }
  return counts;
}

TreeUnits UnitsOfTree(const std::vector<uint32_t> &levels, bool leavesOutside) {
  TreeUnits u;
  for (uint32_t n : levels) u.whole += n;
  if (leavesOutside && levels.size() > 1) u.lowest = levels.back();
  return u;
}

// What a bundle of trees takes in LDS: of those as deep as its walk all but the last level.
struct BundleUnits {
  uint32_t lds = 0;
  uint32_t outside = 0; // leaves that stay out of it
};
BundleUnits UnitsOfBundle(const int32_t *trees, size_t count, const std::vector<int32_t> &depth, const std::vector<TreeUnits> &units) {
  int32_t deepest = 0;
  for (size_t k = 0; k < count; ++k)
    if (trees[k] >= 0) deepest = std::max(deepest, depth[(size_t)trees[k]]);
  BundleUnits b;
  for (size_t k = 0; k < count; ++k) {
    if (trees[k] < 0) continue;
    const TreeUnits &u = units[(size_t)trees[k]];
    const uint32_t lowest = depth[(size_t)trees[k]] == deepest ? u.lowest : 0u;
    b.lds += u.whole - lowest;
    b.outside += lowest;
  }
  return b;
}
// Whether nodes in LDS and leaves outside (4 bytes each), whole 16-byte pieces of either, keep 16-bit addresses.
bool AddressesFit(uint32_t ldsUnits, uint32_t outside) {
  return ((ldsUnits * kNodeBytes + 15u) & ~15u) + ((outside * 4u + 15u) & ~15u) <= 0x10000u;
}

PackedModel PackPlan(const Forest &input, const LaunchPlan &plan, const HitCountProfile *profile, const std::vector<int32_t> *cuts);
bool OwnClassRounds(const Forest &forest, const LaunchPlan &plan, const std::vector<int32_t> &depth, const std::vector<TreeUnits> &units,
                    const std::vector<int32_t> &order, std::vector<std::vector<int32_t>> *rounds);
// Trees order[first], ..., order[first + count - 1] are a bundle of tree group `group`.
struct BundleTrees {
  int32_t group;
  size_t first;
  int32_t count;
};
std::vector<BundleTrees> LayOutGroups(const Forest &forest, const LaunchPlan &plan, const std::vector<int32_t> &depth,
                                      const std::vector<TreeUnits> &units, uint32_t tileUnits, const std::vector<int32_t> &order);
}

namespace {
// The plan with the group sizes that PackForest tries, in that order: the first only if it makes classes the tree threads' own.
std::vector<LaunchPlan> GroupSizes(const LaunchPlan &plan) {
  std::vector<LaunchPlan> tried(plan.ownGroupBytes > 0 ? 2 : 1, plan);
  if (plan.ownGroupBytes > 0) tried[0].groupBytes = plan.ownGroupBytes;
  return tried;
}

// What PackForest goes by of a scalar plan without a profile: the trees' depths and sizes, in its order.
struct PlainTrees {
  std::vector<int32_t> depth, order;
  std::vector<TreeUnits> units;
  PlainTrees(const Forest &forest, const LaunchPlan &plan) : depth(forest.trees.size()), order(forest.trees.size()), units(forest.trees.size()) {
    const bool outside = LeavesOutside(forest, plan);
    for (size_t t = 0; t < forest.trees.size(); ++t) {
      const std::vector<uint32_t> levels = NodesPerLevel(forest.trees[t]);
      depth[t] = (int32_t)levels.size() - 1;
      units[t] = UnitsOfTree(levels, outside);
    }
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
      const int32_t ca = forest.numClasses > 0 ? forest.trees[(size_t)a].classId : 0, cb = forest.numClasses > 0 ? forest.trees[(size_t)b].classId : 0;
      return ca != cb ? ca < cb : depth[(size_t)a] < depth[(size_t)b];
    });
  }
};
} // namespace

bool PacksOwnClasses(const Forest &forest, const LaunchPlan &plan) {
  for (const LaunchPlan &tried : GroupSizes(plan)) {
    const PlainTrees trees(forest, tried);
    std::vector<std::vector<int32_t>> rounds;
    if (OwnClassRounds(forest, tried, trees.depth, trees.units, trees.order, &rounds)) return true;
  }
  return false;
}

int64_t TreeBytesInLds(const Forest &forest, bool leavesOutside) {
  int64_t total = 0;
  for (const Tree &tree : forest.trees) {
    const TreeUnits u = UnitsOfTree(NodesPerLevel(tree), leavesOutside);
    total += u.whole - u.lowest;
  }
  return total * kNodeBytes;
}

// What stays out of LDS makes room for more trees between two barriers and takes the leaf reads off the LDS pipes, and costs a
// gather from L2 per tree.  2^20 rows x 1000 trees of depth 8 (30 % of the nodes are such leaves) 27 groups and 16: 1162 -> 1069
// us; 800 complete trees of depth 6 in 8 classes (half of the nodes) 50 and 25: 849 -> 790.  Not where their bytes are no group
// less: one group either way, 338838 rows x 52 trees of depth 5 22.3 and 22.9, 32 slices of a group, 4096 rows x 1000 trees 12.8 and
// 13.4; nor for the few leaves of skewed trees: 800 of depth 12 in 20 groups and 17 1213 and 1239.
// Between: a 26 % share, 12 groups and 9, 1005 -> 959 us; 28 %, 6 and 4, 86.5 -> 85.0; 29 %, 21 and 14, 1061 -> 989; 35 %, 18 and 12, 1072 ->
// 981; at 19 %, with rows of all kinds through skewed trees, 27 groups and 20 would win too: 1132 and 1086.
// By bytes and not by groups as packed: those can come to as many (a group's addresses reach 64 KB with the leaves outside, and tree
// threads take whole rounds of bundles), and yet half of the copies and the leaf reads are saved.  33 such forests, inside and outside,
// 2 to 41 groups and 50 to 900 trees: complete trees 0.90 to 1.01 of the time (28 groups 139.0 -> 125.5, 41 491 -> 462, 2 339 and 342), shares of
// 26 to 44 % 0.95 to 1.025 (3 groups 445 -> 428, 2 80 -> 78; 2 groups of 163 features 180 -> 184, of 274 47.8 -> 48.8), 0.99 in the mean.
bool LeavesOutside(const Forest &forest, const LaunchPlan &plan) {
  if (plan.kernel != LaunchPlan::Kernel::kRowParallelLds || plan.WalkTile() > 1 || plan.deferTails || plan.quantizedRows || plan.rankRows16)
    return false;
  const int64_t inside = TreeBytesInLds(forest, false), without = TreeBytesInLds(forest, true);
  const auto groups = [&](int64_t bytes) { return std::max<int64_t>(1, (bytes + plan.groupBytes - 1) / plan.groupBytes); };
  const auto turns = [&](int64_t bytes) { return (groups(bytes) + plan.treeSlices - 1) / plan.treeSlices; };
  return without * 5 < inside * 4 && groups(without) >= plan.treeSlices && turns(without) < turns(inside);
}

int32_t CountTreeGroups(const Forest &forest, const LaunchPlan &plan) {
  const PlainTrees trees(forest, plan);
  const std::vector<BundleTrees> bundles = LayOutGroups(forest, plan, trees.depth, trees.units, 1, trees.order);
  return bundles.empty() ? 1 : bundles.back().group + 1;
}

PackedModel PackForest(const Forest &forest, const LaunchPlan &plan, const HitCountProfile *profile) {
  return PackPlan(forest, plan, profile, nullptr);
}

PackedModel PackWithCuts(const Forest &forest, const LaunchPlan &plan, const std::vector<int32_t> &cuts) {
  if (!plan.deferTails || cuts.size() != forest.trees.size()) throw Error("cut levels need a plan with deferred tails and one per tree");
  return PackPlan(forest, plan, nullptr, &cuts);
}

namespace {
// Classes of the tree threads' own: rounds of a bundle for every tree thread, class c's on thread c % treeThreads.  Against them
// stand the classes one after the other, each dealt over all tree threads, which meet at its end: that costs as much as about
// 20 levels of a tree thread.  2^20 rows x 54 features, 800 trees of depth 6, four tree threads, levels of a tree thread that way
// and this, and what was measured: 8 classes 1504 and 1200, 916 and 847 us; 12 1680 and 1224, 969 and 862; 11 1540 and 1368,
// 955 and 894; 7 1484 and 1392, 917 and 910; 10 1400 and 1440, 862 and 890; 9 1476 and 1656, 941 and 957; 6 1416 and 1632, 898
// and 949; 5 1300 and 1920, 853 and 1015.  `order`: by class.  False: the classes meet.
bool OwnClassRounds(const Forest &forest, const LaunchPlan &plan, const std::vector<int32_t> &depth, const std::vector<TreeUnits> &units,
                    const std::vector<int32_t> &order, std::vector<std::vector<int32_t>> *rounds) {
  if (forest.numClasses < 2 || plan.treeThreads < 2 || plan.kernel != LaunchPlan::Kernel::kRowParallelLds || order.empty()) return false;
  const size_t TT = (size_t)plan.treeThreads, C = (size_t)forest.numClasses;
  const int K = plan.interleave;
  const uint32_t groupCapacity = (uint32_t)plan.groupBytes / kNodeBytes;
  std::vector<std::vector<int32_t>> ofClass(C);
  for (int32_t t : order) ofClass[(size_t)forest.trees[(size_t)t].classId].push_back(t);
  double levels = 0.0;
  for (int32_t d : depth) levels += d;
  const double bundleLevels = K * levels / (double)forest.trees.size();
  double meeting = 0.0;
  size_t largest = 0;
  for (auto &trees : ofClass) {
    meeting += (double)((trees.size() + TT * K - 1) / (TT * K)) * bundleLevels + 20.0;
    largest = std::max(largest, trees.size());
  }
  for (size_t c0 = 0; c0 < C; c0 += TT) {
    size_t most = 0;
    for (size_t c = c0; c < std::min(C, c0 + TT); ++c) most = std::max(most, (ofClass[c].size() + K - 1) / K);
    for (size_t i = 0; i < most; ++i) {
      std::vector<int32_t> round(TT * K, -1);
      BundleUnits need;
      for (size_t c = c0; c < std::min(C, c0 + TT); ++c) {
        for (size_t k = 0; k < (size_t)K && i * K + k < ofClass[c].size(); ++k) round[(c - c0) * K + k] = ofClass[c][i * K + k];
        const BundleUnits bundle = UnitsOfBundle(&round[(c - c0) * K], (size_t)K, depth, units);
        need.lds += bundle.lds;
        need.outside += bundle.outside;
      }
      if (need.lds + 2 > groupCapacity - 1 || !AddressesFit(need.lds + 2, need.outside)) return false;
      rounds->push_back(std::move(round));
    }
  }
  // Near a tie the threads that wait can lose, with tree slices most.  230 forests of 2 to 16 classes, both ways: without slices
  // 0.34 to 0.98 of the time up to 0.95 of the cost, but 1.04 at 0.92 where all of a class is one round of bundles (74 trees, five
  // classes); with slices up to 1.01 below 0.81 of the cost, 1.10 at 0.84.
  const double share = plan.treeSlices > 1 ? 0.81 : largest <= TT * K ? 0.9 : 0.95;
  return (double)rounds->size() * bundleLevels < meeting * share;
}

// Bundles of up to K consecutive trees of one class, in groups of what fits the plan's group size.  Tree threads take bundles
// round-robin: when more trees follow, a group ends on a multiple of treeThreads bundles so that no thread idles through a last
// partial round.
std::vector<BundleTrees> LayOutGroups(const Forest &forest, const LaunchPlan &plan, const std::vector<int32_t> &depth,
                                      const std::vector<TreeUnits> &units, uint32_t tileUnits, const std::vector<int32_t> &order) {
  const uint32_t groupCapacity = (uint32_t)plan.groupBytes / kNodeBytes;
  const size_t multiple = plan.kernel == LaunchPlan::Kernel::kRowParallelLds ? (size_t)plan.treeThreads : 1;
  std::vector<BundleTrees> out;
  size_t next = 0;
  for (int32_t group = 0; next < order.size(); ++group) {
    const size_t begin = out.size();
    uint32_t used = tileUnits, usedOutside = 0; // the null leaf
    while (next < order.size()) {
      const int32_t cls = forest.numClasses > 0 ? forest.trees[order[next]].classId : 0;
      int32_t count = 0;
      BundleUnits bundle;
      while (count < plan.interleave && next + count < order.size()) {
        const int32_t t = order[next + count];
        const int32_t c = forest.numClasses > 0 ? forest.trees[t].classId : 0;
        if (c != cls) break;
        if (units[t].whole + 2 * tileUnits > groupCapacity)
          throw Error("a tree of " + std::to_string(forest.trees[t].NumNodes()) + " nodes does not fit one LDS tree group");
        const BundleUnits with = UnitsOfBundle(&order[next], (size_t)count + 1, depth, units);
        if (used + with.lds > groupCapacity - 1 || !AddressesFit(used + with.lds, usedOutside + with.outside)) break; // (one spare unit keeps room for the alignment pad)
        bundle = with;
        ++count;
      }
      if (count == 0) break; // group full
      used += bundle.lds;
      usedOutside += bundle.outside;
      out.push_back(BundleTrees{group, next, count});
      next += (size_t)count;
    }
    if (out.size() == begin) throw Error("internal error: empty tree group");
    const size_t bundles = out.size() - begin;
    if (next < order.size() && multiple > 1 && bundles > multiple && bundles % multiple != 0) {
      const size_t keep = begin + bundles - bundles % multiple;
      next = out[keep].first;
      out.resize(keep);
    }
  }
  return out;
}

constexpr uint32_t kPeeledTailNodes = 1u << 20; // below the cuts of a plan with a profile (8 MB: they stay in the caches)

PackedModel PackPlan(const Forest &input, const LaunchPlan &asked, const HitCountProfile *profile, const std::vector<int32_t> *cuts) {
  LaunchPlan plan = asked; // (of its groups' two sizes the one that is taken, once that is known)
  // Plans also come out of files: every field is brought into its range before anything is computed from it.
  if (plan.kernel != LaunchPlan::Kernel::kRowParallelLds && plan.kernel != LaunchPlan::Kernel::kTreeParallel &&
      plan.kernel != LaunchPlan::Kernel::kGlobalWalk)
    throw Error("launch plan names no kernel");
  if (plan.rowsPerBlock < 1 || plan.rowsPerBlock > 1024 || plan.treeThreads < 1 || plan.treeThreads > 1024 || plan.treeLanes < 1 ||
      plan.treeLanes > 1024)
    throw Error("launch plan: rows per block, tree threads and tree lanes must be in [1, 1024]");
  if (plan.treeSlices < 1 || plan.treeSlices > 65535) throw Error("launch plan: tree slices must be in [1, 65535]");
  if (plan.tiling < 0 || plan.tiling > 2) throw Error("launch plan: tiling type must be 0, 1 or 2");
  const Forest forest = NormalizeToLessThan(input);
  if (profile && profile->hits.size() != forest.trees.size()) throw Error("hit-count profile does not match the forest");
  if (plan.kernel == LaunchPlan::Kernel::kGlobalWalk) {
    if (plan.WalkTile() > 1) throw Error("tile sizes above 1 need the row-parallel LDS kernel; this forest has a tree too big for LDS");
    return PackForGlobalWalk(forest, plan);
  }
  const int K = plan.interleave;
  if (K < 1 || K > kMaxInterleave || (K & (K - 1))) throw Error("interleave must be 1, 2, 4 or 8");
  if (plan.kernel == LaunchPlan::Kernel::kRowParallelLds) {
    if (plan.rowsPerBlock < 64 || (plan.rowsPerBlock & (plan.rowsPerBlock - 1)) || plan.rowsPerBlock > 1024)
      throw Error("rowsPerBlock must be a power of two in [64, 1024]");
    if (plan.treeThreads < 1 || plan.ThreadsPerBlock() > 1024)
      throw Error("rowsPerBlock * treeThreads must not exceed 1024 lanes");
  } else {
    if (plan.treeLanes < 1 || (plan.treeLanes & (plan.treeLanes - 1)) || plan.rowsPerBlock < 1 ||
        plan.ThreadsPerBlock() > 1024 || plan.ThreadsPerBlock() % 64 != 0)
      throw Error("tree-parallel plan needs a power-of-two treeLanes and a block of 64..1024 lanes");
    if (plan.treeLanes < 64 && 64 % plan.treeLanes != 0) throw Error("treeLanes must divide 64");
  }
  if (plan.groupBytes > 256 * plan.ThreadsPerBlock())
    throw Error("groupBytes must not exceed 256 bytes per lane of the block (group prefetch registers)");
  if (plan.groupBytes < 1024 || plan.groupBytes > 65536) throw Error("groupBytes must be in [1024, 65536]");
  if (plan.ownGroupBytes != 0 && (plan.kernel != LaunchPlan::Kernel::kRowParallelLds || forest.numClasses < 2 || plan.ownGroupBytes < plan.groupBytes ||
                                  plan.ownGroupBytes > std::min(65536, 256 * plan.ThreadsPerBlock())))
    throw Error("launch plan: groups of the tree threads' own classes are no smaller than others and keep their limits");

  if (plan.quantizedRows && (plan.kernel != LaunchPlan::Kernel::kRowParallelLds || plan.rowsPerBlock != 64))
    throw Error("rank-quantised rows need the row-parallel kernel with 64 rows per block");
  if (plan.rankRows16 && (plan.kernel != LaunchPlan::Kernel::kRowParallelLds || plan.quantizedRows || plan.featureOffsetInWords))
    throw Error("two-byte rank rows need the row-parallel kernel (and exclude one-byte ranks and word offsets)");
  if (plan.tileSize < 1 || plan.tileSize > kMaxTileSize)
    throw Error("tile size " + std::to_string(plan.tileSize) + " is not supported: the device kernels walk tiles of 1 to " +
                std::to_string(kMaxTileSize) + " nodes");
  const int T = plan.WalkTile();
  if (plan.deferTails && (plan.kernel != LaunchPlan::Kernel::kRowParallelLds || T != 1 || plan.quantizedRows || plan.rankRows16 ||
                          plan.featureOffsetInWords || forest.numClasses > 0 || !(profile || cuts)))
    throw Error("deferred tails need a profile and the scalar row-parallel kernel on float32 rows of a model without classes");
  if (T > 1 && (plan.kernel != LaunchPlan::Kernel::kRowParallelLds || plan.quantizedRows || plan.rankRows16))
    throw Error("tile sizes above 1 need the row-parallel kernel on float32 rows");
  if (T > 1 && (plan.featureOffsetInWords || (int64_t)(forest.numFeatures + 1) * plan.rowsPerBlock * 4 > 0x10000))
    throw Error("tile sizes above 1 need a row tile below 64 KB (tiles hold byte offsets): fewer rows per block");

  PackedModel pm;
  pm.plan = asked;
  pm.numFeatures = forest.numFeatures;
  pm.numClasses = forest.numClasses;
  pm.numTrees = (int32_t)forest.trees.size();
  if (plan.deferTails) { // tail node 0: a leaf of value 0, what a lane without a queue entry walks
    pm.tailNodes.push_back(DeviceNode{0.0f, (0u << kTailFeatureBits) | (uint32_t)forest.numFeatures});
    pm.tailOrigin.push_back(-1);
  }
  const uint64_t padOffset = pm.PadFeatureOffset();
  if (padOffset > 0xFFFFu)
    throw Error("feature offsets do not fit 16 bits for this rowsPerBlock / feature count");
  const uint32_t featureStride = plan.FeatureStride();
  if (plan.rankRows16 && pm.RowTileBytes() > 0x10000u) throw Error("two-byte rank rows: the row tile must stay below 64 KB (byte offsets)");
  const uint32_t tileUnits = TileBytes(T) / kNodeBytes;                    // units per tile (1 for scalar nodes)

  // Rank quantisation: x < t_j  <=>  #{t : t <= x} <= j for the sorted distinct thresholds t_0 < t_1 < ...
  // of the feature, so an internal node stores j and the kernel compares the row's one-byte rank with it.
  std::vector<std::vector<float>> ranks;
  if (plan.quantizedRows) {
    ranks = ThresholdsPerFeature(forest);
    size_t most = 0;
    for (auto &v : ranks) most = std::max(most, v.size());
    if (most > 254) throw Error("a feature has more than 254 distinct thresholds: rows cannot be rank-quantised to bytes");
    int32_t depth = 1;
    while ((size_t)depth < most) depth = depth * 2 + 1; // 2^n - 1 >= most
    pm.binTableDepth = depth;
    // features per block of the binning kernel: one per lane of a wave
    const int32_t chunk = 64;
    pm.binChunkFeatures = chunk;
    const int32_t chunks = (forest.numFeatures + chunk - 1) / chunk;
    pm.binThresholds.assign((size_t)chunks * depth * chunk, std::numeric_limits<float>::infinity());
    for (int32_t f = 0; f < forest.numFeatures; ++f)
      for (size_t k = 0; k < ranks[f].size(); ++k)
        pm.binThresholds[((size_t)(f / chunk) * depth + k) * chunk + (f % chunk)] = ranks[f][k];
  }

  if (plan.rankRows16) {
    ranks = ThresholdsPerFeature(forest);
    // LDS of one block of the ranking kernel: the chunk's tables and a staging tile of 1025 floats per feature of
    // the chunk (two blocks per compute unit)
    constexpr size_t kChunkBytes = 76 * 1024, kStageBytesPerFeature = 1025 * 4;
    pm.rankFeatures.resize((size_t)((forest.numFeatures + 2) / 2) * 2); // every slot of the tile, the pad feature's included
    auto tableEntries = [&](size_t f) -> size_t {
      if (f >= ranks.size() || ranks[f].empty()) return 0;
      size_t entries = 1;
      while (entries < ranks[f].size()) entries = entries * 2 + 1; // 2^n - 1 >= thresholds
      return entries;
    };
    for (size_t f = 0; f < ranks.size(); ++f)
      if (ranks[f].size() > 65534) throw Error("a feature has more than 65534 distinct thresholds: rows cannot be ranked in two bytes");
    size_t f = 0;
    while (f < pm.rankFeatures.size()) {
      RankChunkDesc chunk{(uint32_t)f, 0, (uint32_t)pm.rankTables.size(), 0};
      size_t entries = 0;
      while (f < pm.rankFeatures.size()) {
        const size_t pairEntries = tableEntries(f) + tableEntries(f + 1);
        if (pairEntries * 4 + 2 * kStageBytesPerFeature > 150 * 1024) throw Error("the thresholds of one feature pair do not fit the ranking kernel's LDS");
        if (chunk.numFeatures > 0 && (entries + pairEntries) * 4 + (chunk.numFeatures + 2) * kStageBytesPerFeature > kChunkBytes) break;
        for (size_t g = f; g < f + 2; ++g) {
          const size_t n = tableEntries(g);
          uint32_t levels = 0;
          while (((size_t)1 << levels) - 1 < n) ++levels;
          pm.rankFeatures[g] = RankFeatureDesc{(uint32_t)entries, levels};
          // breadth-first order of the complete search tree over the sorted thresholds (+inf beyond the last)
          std::vector<float> bfs(n, std::numeric_limits<float>::infinity());
          std::function<void(size_t, size_t, size_t)> fill = [&](size_t node, size_t lo, size_t hi) { // keys [lo, hi)
            if (node >= n) return;
            const size_t mid = lo + (hi - lo) / 2;
            if (mid < ranks[g].size()) bfs[node] = ranks[g][mid];
            fill(2 * node + 1, lo, mid);
            fill(2 * node + 2, mid + 1, hi);
          };
          fill(0, 0, n);
          pm.rankTables.insert(pm.rankTables.end(), bfs.begin(), bfs.end());
          entries += n;
        }
        chunk.numFeatures += 2;
        f += 2;
      }
      chunk.tableEntries = (uint32_t)entries;
      pm.rankChunks.push_back(chunk);
    }
    pm.rankThresholds = ranks;
  }

  // Per tree: its size in the packed layout, the steps of a lock-step walk, and the steps after which the walk
  // starts looking whether any lane still moves (walk peeling; equal to the depth when there is no tail).
  const size_t numTrees = forest.trees.size();
  std::vector<TiledTree> tiled(T > 1 ? numTrees : 0);
  std::vector<int32_t> depth(numTrees), peel(numTrees);
  std::vector<int32_t> fullDepth(numTrees, 0); // deferred tails: the tree's own depth (depth[] is then where its walk stops)
  int64_t tailBudget = plan.deferTails && forest.numFeatures + 1 < (1 << kTailFeatureBits) ? (int64_t)(cuts ? kMaxTailNodes : kPeeledTailNodes) - 1 : 0;
  std::vector<TreeUnits> units(numTrees);
  std::vector<std::vector<uint32_t>> levels(T > 1 ? 0 : numTrees); // (of the nodes that walks reach: pruned models keep others)
  for (size_t t = 0; t < numTrees; ++t) {
    const Tree &tree = forest.trees[t];
    const std::vector<int64_t> *hits = profile ? &profile->hits[t] : nullptr;
    std::vector<int32_t> leafLevel(tree.NumNodes(), -1);
    std::vector<int32_t> nodeLevel; // scalar nodes: the level of every node
    if (T > 1) {
      tiled[t] = TileTree(tree, T, plan.tiling, hits);
      depth[t] = tiled[t].depth;
      units[t].whole = (uint32_t)tiled[t].tiles.size() * tileUnits;
      pm.treesTiledByProfile += tiled[t].byProfile ? 1 : 0;
      pm.maxTileHops = std::max(pm.maxTileHops, tiled[t].hops);
      for (const TileInfo &tile : tiled[t].tiles)
        if (tile.count == 0) leafLevel[tile.leafNode] = tile.level;
    } else {
      depth[t] = tree.Depth();
      levels[t] = NodesPerLevel(tree);
      units[t] = UnitsOfTree(levels[t], false);
      std::vector<int32_t> stack{0};
      leafLevel[0] = 0;
      while (!stack.empty()) { // (the level of every node; only the leaves' entries are used)
        const int32_t n = stack.back();
        stack.pop_back();
        if (tree.IsLeaf(n)) continue;
        leafLevel[tree.left[n]] = leafLevel[tree.right[n]] = leafLevel[n] + 1;
        stack.push_back(tree.left[n]);
        stack.push_back(tree.right[n]);
      }
      nodeLevel = leafLevel;
      for (size_t i = 0; i < tree.NumNodes(); ++i)
        if (!tree.IsLeaf((int32_t)i)) leafLevel[i] = -1;
    }
    peel[t] = plan.peelWalks && hits ? PeelDepth(*hits, leafLevel, depth[t]) : depth[t];
    fullDepth[t] = depth[t];
    int32_t cut = cuts ? std::min((*cuts)[t], depth[t]) : depth[t];
    double queued = 0.0; // (of the profiled rows, by the profile)
    if (plan.deferTails && !cuts) {
      // Where the lock-step walk of this tree stops.  Costs in cycles of a compute unit per 64 rows: a lock-step
      // level is a node read (2.5 cycles while the level has at most 32 nodes, 4.3 for 64, 6.0 beyond) and a
      // feature read (2.4), as measured on MI355X; a deferred walk costs 20 to queue, fetch and hand back plus 20
      // per step down to the deepest leaf below the stub (a wave of 64 queue entries runs to the deepest of them),
      // and the stub test costs every row of the tree 2: the values that, of those tried (6 to 150 per step), gave
      // the shortest kernel times on two models of 1000 and 800 trees.
      std::vector<double> alive((size_t)depth[t] + 1, 0.0);
      {
        std::vector<std::pair<int32_t, int32_t>> stack{{0, 0}};
        while (!stack.empty()) {
          auto [n, level] = stack.back();
          stack.pop_back();
          if (tree.IsLeaf(n)) continue;
          alive[(size_t)level] += (*hits)[0] > 0 ? (double)(*hits)[n] / (double)(*hits)[0] : 1.0;
          stack.push_back({tree.left[n], level + 1});
          stack.push_back({tree.right[n], level + 1});
        }
      }
      auto levelCost = [](int32_t d) { return (d <= 5 ? 2.5 : d == 6 ? 4.3 : 6.0) + 2.4; };
      double whole = 0.0;
      for (int32_t d = 0; d < depth[t]; ++d) whole += levelCost(d);
      double best = whole, head = 0.0;
      for (int32_t d = 1; d < depth[t]; ++d) {
        head += levelCost(d - 1);
        const double cost = head + 2.0 + alive[(size_t)d] * ((depth[t] - d) * 20.0 + 20.0);
        if (cost < best && cost < 0.92 * whole) best = cost, cut = d;
      }
      queued = alive[(size_t)cut];
    }
    if (cut < depth[t]) {
      bool nanLeaf = false; // (a NaN is what marks a stub)
      for (size_t i = 0; i < tree.NumNodes(); ++i) nanLeaf = nanLeaf || (tree.IsLeaf((int32_t)i) && tree.value[i] != tree.value[i]);
      uint32_t above = 0; // the top of the tree, the cut level's internal nodes as stubs
      int64_t tails = 0;  // those internal nodes again, and all below them
      for (size_t i = 0; i < tree.NumNodes(); ++i) {
        if (nodeLevel[i] >= 0 && nodeLevel[i] <= cut) ++above;
        if (nodeLevel[i] > cut || (nodeLevel[i] == cut && !tree.IsLeaf((int32_t)i))) ++tails;
      }
      if (tails <= tailBudget && !nanLeaf) {
        tailBudget -= tails;
        units[t].whole = above;
        depth[t] = cut;
        peel[t] = cut;
        pm.treesDeferred += 1;
        pm.deferredEntriesPerRow += queued;
      }
    }
    pm.lockStepSteps += depth[t];
    if (hits && (*hits)[0] > 0) {
      double steps = 0.0;
      for (size_t i = 0; i < tree.NumNodes(); ++i)
        if (leafLevel[i] >= 0) steps += (double)(*hits)[i] * leafLevel[i];
      pm.profiledSteps += steps / (double)(*hits)[0];
    }
  }

  // Order: class, then depth (the reference sorts by depth for its GPU schedules,
  // src/mlir/GPUAutoSchedule.cpp:115-122); stable so equal keys keep model order.
  std::vector<int32_t> order(numTrees);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
    int32_t ca = forest.numClasses > 0 ? forest.trees[a].classId : 0;
    int32_t cb = forest.numClasses > 0 ? forest.trees[b].classId : 0;
    if (ca != cb) return ca < cb;
    if (depth[a] != depth[b]) return depth[a] < depth[b];
    return peel[a] < peel[b];
  });

  // The groups' size, what stays out of them, and whose the classes are.
  std::vector<std::vector<int32_t>> rounds; // classes of the tree threads' own: treeThreads * K trees each, -1: none
  for (const LaunchPlan &tried : GroupSizes(asked)) {
    plan = tried;
    pm.groupBytes = plan.groupBytes;
    pm.leavesOutside = LeavesOutside(forest, plan);
    if (T > 1) continue;
    for (size_t t = 0; t < numTrees && !plan.deferTails; ++t) units[t] = UnitsOfTree(levels[t], pm.leavesOutside);
    rounds.clear();
    pm.ownClasses = OwnClassRounds(forest, plan, depth, units, order, &rounds);
    if (pm.ownClasses) break;
  }
  const uint32_t groupCapacity = (uint32_t)plan.groupBytes / kNodeBytes; // in 8-byte units

  const auto pushUnit = [&](const DeviceNode &node, int32_t origin, int32_t second = -1) {
    pm.nodes.push_back(node);
    pm.nodeOrigin.push_back(origin);
    pm.nodeOrigin.push_back(second);
  };
  // The null leaf that padding trees of a bundle point at: a leaf of value 0 at address 0 of every group.
  auto pushNullLeaf = [&]() {
    if (T > 1) {
      Tree nullTree;
      nullTree.value = {0.0f};
      nullTree.feature = {0};
      nullTree.left = nullTree.right = {-1};
      TileInfo leaf;
      leaf.leafNode = 0;
      std::vector<unsigned char> bytes(TileBytes(T));
      EmitTile(nullTree, leaf, T, 0, 0, featureStride, (uint32_t)padOffset, bytes.data());
      for (uint32_t u = 0; u < tileUnits; ++u) {
        DeviceNode unit;
        std::memcpy(&unit, bytes.data() + u * kNodeBytes, kNodeBytes);
        pushUnit(unit, -1);
      }
    } else {
      pushUnit(DeviceNode{0.0f, NodeMeta(0, (uint32_t)padOffset)}, -1);
    }
  };
  auto openGroup = [&]() {
    DeviceGroup g{};
    g.nodeBegin = (uint32_t)pm.nodes.size();
    g.bundleBegin = (uint32_t)pm.bundles.size();
    pm.groups.push_back(g);
    pushNullLeaf();
  };
  // Leaves of the group that stay out of LDS, and the nodes whose children they are (which count from the first of them until it
  // is known where that lies).
  std::vector<float> outside;
  std::vector<int32_t> outsideOrigin;
  std::vector<size_t> aboveOutside;
  auto pad = [&]() { // whole 16-byte pieces
    if ((pm.nodes.size() - pm.groups.back().nodeBegin) & 1) pushUnit(DeviceNode{0.0f, NodeMeta(0, (uint32_t)padOffset)}, -1);
  };
  auto closeGroup = [&]() {
    DeviceGroup &g = pm.groups.back();
    pad();
    g.nodeCount = (uint32_t)pm.nodes.size() - g.nodeBegin;
    for (size_t n : aboveOutside) pm.nodes[n].meta = NodeMeta(MetaChild(pm.nodes[n].meta) + g.nodeCount * kNodeBytes, MetaFeature(pm.nodes[n].meta));
    if (outside.size() & 1) {
      outside.push_back(0.0f);
      outsideOrigin.push_back(-1);
    }
    for (size_t i = 0; i < outside.size(); i += 2) {
      DeviceNode two;
      std::memcpy(&two, &outside[i], sizeof(two));
      pushUnit(two, outsideOrigin[i], outsideOrigin[i + 1]);
    }
    outside.clear();
    outsideOrigin.clear();
    aboveOutside.clear();
    pad();
    g.imageCount = (uint32_t)pm.nodes.size() - g.nodeBegin;
    if (g.imageCount * kNodeBytes > 0x10000u) throw Error("internal error: tree group beyond 16-bit addresses");
    g.bundleCount = (uint32_t)pm.bundles.size() - g.bundleBegin;
    for (uint32_t b = g.bundleBegin; b < pm.bundles.size(); ++b)
      for (int k = 0; k < K; ++k) pm.bundleRoots.push_back(pm.nodes[g.nodeBegin + pm.bundles[b].root[k] / kNodeBytes]);
    g.uniformClass = 0;
    if (g.bundleCount > 0) {
      const uint32_t first = pm.bundles[g.bundleBegin].classId;
      bool uniform = true;
      for (uint32_t b = 1; b < g.bundleCount; ++b) uniform = uniform && pm.bundles[g.bundleBegin + b].classId == first;
      if (uniform) g.uniformClass = first + 1;
    }
    pm.maxGroupNodes = std::max(pm.maxGroupNodes, g.nodeCount);
  };
  // Writes tree t with its first unit at unit `base` of the current group, to be walked for `steps` levels.
  auto emitTree = [&](int32_t t, uint32_t base, int32_t steps) {
    const Tree &tree = forest.trees[t];
    if (T > 1) {
      std::vector<unsigned char> bytes(TileBytes(T));
      for (size_t ti = 0; ti < tiled[t].tiles.size(); ++ti) {
        const TileInfo &tile = tiled[t].tiles[ti];
        EmitTile(tree, tile, T, base * kNodeBytes, ti, featureStride, (uint32_t)padOffset, bytes.data());
        for (uint32_t u = 0; u < tileUnits; ++u) {
          DeviceNode unit;
          std::memcpy(&unit, bytes.data() + u * kNodeBytes, kNodeBytes);
          pushUnit(unit, u == 0 ? (tile.count == 0 ? tile.leafNode : tile.members[0]) : -1);
        }
      }
      return;
    }
    if (plan.deferTails && depth[t] < fullDepth[t]) {
      // The walk of this tree stops at level depth[t]: the internal nodes of that level are represented by stubs
      // (a NaN whose payload is the index of the node itself in the tail array); their subtrees go to the tail
      // array in global memory, each in level order with siblings adjacent.
      const int32_t cut = depth[t];
      std::vector<int32_t> top, cutNodes, where(tree.NumNodes(), -1);
      {
        std::vector<std::pair<int32_t, int32_t>> queue{{0, 0}};
        for (size_t head = 0; head < queue.size(); ++head) {
          auto [n, level] = queue[head];
          where[n] = (int32_t)top.size();
          top.push_back(n);
          if (tree.IsLeaf(n)) continue;
          if (level == cut) { cutNodes.push_back(n); continue; }
          queue.push_back({tree.left[n], level + 1});
          queue.push_back({tree.right[n], level + 1});
        }
      }
      if (top.size() != units[t].whole) throw Error("internal error: deferred tree size out of step");
      std::vector<uint32_t> tailIndex(tree.NumNodes(), 0);
      for (int32_t first : cutNodes) {
        std::vector<int32_t> queue{first};
        for (size_t head = 0; head < queue.size(); ++head) {
          const int32_t n = queue[head];
          if (!tree.IsLeaf(n)) { queue.push_back(tree.left[n]); queue.push_back(tree.right[n]); }
        }
        const uint32_t begin = (uint32_t)pm.tailNodes.size();
        if ((size_t)begin + queue.size() > kMaxTailNodes) throw Error("internal error: tail array overflow");
        for (size_t i = 0; i < queue.size(); ++i) tailIndex[queue[i]] = begin + (uint32_t)i;
        for (int32_t n : queue) {
          DeviceNode dn;
          dn.value = tree.value[n];
          if (tree.IsLeaf(n)) {
            dn.meta = (tailIndex[n] << kTailFeatureBits) | (uint32_t)forest.numFeatures; // stays put: the pad feature holds -inf
          } else {
            if (tailIndex[tree.right[n]] != tailIndex[tree.left[n]] + 1) throw Error("internal error: siblings not adjacent");
            dn.meta = (tailIndex[tree.left[n]] << kTailFeatureBits) | (uint32_t)tree.feature[n];
          }
          pm.tailNodes.push_back(dn);
          pm.tailOrigin.push_back(n);
        }
      }
      for (size_t i = 0; i < top.size(); ++i) {
        const int32_t n = top[i];
        const uint32_t self = (base + (uint32_t)i) * kNodeBytes;
        DeviceNode dn;
        if (tree.IsLeaf(n)) {
          dn.value = tree.value[n];
          dn.meta = NodeMeta(self, (uint32_t)padOffset);
        } else if (tailIndex[n] != 0) { // a stub: NaN compares false, so the walk takes the "right" child: the stub itself
          const uint32_t bits = kStubValueBits | tailIndex[n];
          std::memcpy(&dn.value, &bits, sizeof(bits));
          dn.meta = NodeMeta(self - kNodeBytes, (uint32_t)padOffset);
        } else {
          dn.value = tree.value[n];
          if (where[tree.right[n]] != where[tree.left[n]] + 1) throw Error("internal error: siblings not adjacent");
          dn.meta = NodeMeta((base + (uint32_t)where[tree.left[n]]) * kNodeBytes, plan.FeatureOffset((uint32_t)tree.feature[n]));
        }
        pushUnit(dn, n);
      }
      pm.maxTailDepth = std::max<uint32_t>(pm.maxTailDepth, (uint32_t)(fullDepth[t] - cut));
      return;
    }
    const LevelOrder lo = MakeLevelOrder(tree);
    const size_t inside = lo.order.size() - (depth[t] == steps ? units[t].lowest : 0u); // (level order: the last level comes last)
    const size_t firstOutside = outside.size();
    for (size_t i = 0; i < lo.order.size(); ++i) {
      const int32_t n = lo.order[i];
      DeviceNode dn;
      dn.value = tree.value[n];
      if (i >= inside) {
        outside.push_back(tree.value[n]);
        outsideOrigin.push_back(n);
        continue;
      }
      if ((plan.quantizedRows || plan.rankRows16) && !tree.IsLeaf(n)) {
        const auto &sorted = ranks[(size_t)tree.feature[n]];
        const uint32_t j = (uint32_t)(std::lower_bound(sorted.begin(), sorted.end(), tree.value[n]) - sorted.begin());
        static_assert(sizeof(float) == sizeof(uint32_t), "node value holds the rank bit pattern");
        std::memcpy(&dn.value, &j, sizeof(j));
      }
      if (tree.IsLeaf(n)) {
        dn.meta = NodeMeta((base + (uint32_t)i) * kNodeBytes, (uint32_t)padOffset);
      } else {
        const size_t left = (size_t)lo.position[tree.left[n]];
        if (lo.position[tree.right[n]] != lo.position[tree.left[n]] + 1)
          throw Error("internal error: siblings not adjacent");
        const uint32_t child = (uint32_t)(left < inside ? (base + left) * kNodeBytes : (firstOutside + (left - inside)) * 4u);
        if (left >= inside) aboveOutside.push_back(pm.nodes.size());
        dn.meta = NodeMeta(child, plan.FeatureOffset((uint32_t)tree.feature[n]));
      }
      pushUnit(dn, n);
    }
  };

  if (pm.ownClasses) {
    const size_t TT = (size_t)plan.treeThreads;
    for (size_t next = 0; next < rounds.size();) {
      openGroup();
      DeviceGroup &g = pm.groups.back();
      for (; next < rounds.size(); ++next) {
        BundleUnits need;
        for (size_t thread = 0; thread < TT; ++thread) {
          const BundleUnits bundle = UnitsOfBundle(&rounds[next][thread * K], (size_t)K, depth, units);
          need.lds += bundle.lds;
          need.outside += bundle.outside;
        }
        const uint32_t used = (uint32_t)pm.nodes.size() - g.nodeBegin;
        if (need.lds > groupCapacity - 1 - used || !AddressesFit(used + need.lds, (uint32_t)outside.size() + need.outside)) break;
        for (size_t thread = 0; thread < TT; ++thread) {
          DeviceBundle b{};
          b.firstSlot = (uint32_t)pm.slotTree.size();
          for (int k = 0; k < K; ++k) {
            const int32_t t = rounds[next][thread * K + (size_t)k];
            pm.slotTree.push_back(t);
            if (t >= 0) b.depth = b.peelDepth = std::max<uint32_t>(b.depth, (uint32_t)depth[(size_t)t]);
          }
          for (int k = 0; k < K; ++k) {
            const int32_t t = rounds[next][thread * K + (size_t)k];
            if (t < 0) continue; // (root 0: the null leaf)
            const uint32_t base = (uint32_t)pm.nodes.size() - g.nodeBegin;
            b.root[k] = (uint16_t)(base * kNodeBytes);
            emitTree(t, base, (int32_t)b.depth);
          }
          const int32_t any = rounds[next][thread * K];
          // (a bundle without trees keeps its thread's class, the first one's if it had none yet)
          b.classId = any >= 0 ? (uint16_t)forest.trees[(size_t)any].classId
                      : pm.bundles.size() >= TT ? pm.bundles[pm.bundles.size() - TT].classId : (uint16_t)thread;
          pm.bundles.push_back(b);
        }
      }
      closeGroup();
    }
  }

  const std::vector<BundleTrees> laidOut = pm.ownClasses ? std::vector<BundleTrees>() : LayOutGroups(forest, plan, depth, units, tileUnits, order);
  for (size_t at = 0; at < laidOut.size();) {
    openGroup();
    DeviceGroup &g = pm.groups.back();
    for (const int32_t group = laidOut[at].group; at < laidOut.size() && laidOut[at].group == group; ++at) {
      DeviceBundle b{};
      b.classId = (uint16_t)(forest.numClasses > 0 ? forest.trees[order[laidOut[at].first]].classId : 0);
      b.firstSlot = (uint32_t)pm.slotTree.size();
      for (int k = 0; k < laidOut[at].count; ++k) b.depth = std::max<uint32_t>(b.depth, (uint32_t)depth[order[laidOut[at].first + k]]);
      for (int k = 0; k < K; ++k) {
        if (k >= laidOut[at].count) {
          b.root[k] = 0; // null leaf
          pm.slotTree.push_back(-1);
          continue;
        }
        const int32_t t = order[laidOut[at].first + k];
        const uint32_t base = (uint32_t)pm.nodes.size() - g.nodeBegin; // unit index inside the group
        b.root[k] = (uint16_t)(base * kNodeBytes);
        b.peelDepth = std::max<uint32_t>(b.peelDepth, (uint32_t)peel[t]);
        if (plan.deferTails && depth[t] < fullDepth[t]) b.hasStubs = 1;
        pm.slotTree.push_back(t);
        emitTree(t, base, (int32_t)b.depth);
      }
      pm.bundles.push_back(b);
    }
    closeGroup();
  }
  if (pm.groups.empty()) { // a forest without trees still needs one (empty) group
    openGroup();
    closeGroup();
  }
  if (pm.bundleRoots.size() != pm.bundles.size() * (size_t)K) throw Error("internal error: bundle root table out of step");
  return pm;
}
} // namespace

Tree UnpackTree(const PackedModel &pm, int32_t treeIndex) {
  if (pm.plan.WalkTile() > 1) throw Error("tiled models are checked through their walks, not unpacked");
  if (pm.plan.kernel == LaunchPlan::Kernel::kGlobalWalk) {
    for (const DeviceGlobalTree &gt : pm.globalTrees) {
      if (gt.origin != treeIndex) continue;
      Tree tree;
      tree.classId = (int32_t)gt.classId;
      std::vector<uint32_t> queue{gt.root};
      size_t total = 0;
      for (size_t head = 0; head < queue.size(); ++head) {
        const DeviceGlobalNode &dn = pm.globalNodes[queue[head]];
        total = std::max<size_t>(total, (size_t)dn.origin + 1);
        if (dn.feature != kGlobalLeaf) { queue.push_back(dn.left); queue.push_back(dn.left + 1); }
      }
      tree.value.assign(total, 0.f);
      tree.feature.assign(total, 0);
      tree.left.assign(total, -1);
      tree.right.assign(total, -1);
      for (uint32_t q : queue) {
        const DeviceGlobalNode &dn = pm.globalNodes[q];
        tree.value[dn.origin] = dn.value;
        if (dn.feature != kGlobalLeaf) {
          tree.feature[dn.origin] = (int32_t)dn.feature;
          tree.left[dn.origin] = pm.globalNodes[dn.left].origin;
          tree.right[dn.origin] = pm.globalNodes[dn.left + 1].origin;
        }
      }
      return tree;
    }
    throw Error("tree not found in packed model");
  }
  const int K = pm.plan.interleave;
  for (const DeviceGroup &g : pm.groups)
    for (uint32_t bi = g.bundleBegin; bi < g.bundleBegin + g.bundleCount; ++bi)
      for (int k = 0; k < K; ++k) {
        if (pm.slotTree[pm.bundles[bi].firstSlot + k] != treeIndex) continue;
        // walk the packed tree breadth first, restoring original node ids (a stub stands for the node its value
        // field points at)
        // (words of the group's image, whose nodes take two and whose leaves outside LDS one; a stub stands for a node of the
        // tail array, noted as kTailBit | index)
        constexpr uint32_t kTailBit = 0x80000000u;
        auto resolve = [&](uint32_t word) {
          if (word >= g.nodeCount * 2) return word;
          const DeviceNode &dn = pm.nodes[g.nodeBegin + word / 2];
          uint32_t bits;
          std::memcpy(&bits, &dn.value, sizeof(bits));
          const bool stub = pm.plan.deferTails && MetaChild(dn.meta) / kNodeBytes + 1 == word / 2 && (bits & ~kStubIndexMask) == kStubValueBits;
          if (!stub) return word;
          return kTailBit | (bits & kStubIndexMask);
        };
        auto outsideLds = [&](uint32_t q) { return !(q & kTailBit) && q >= g.nodeCount * 2; };
        auto nodeAt = [&](uint32_t q) {
          if (q & kTailBit) return pm.tailNodes[q & ~kTailBit];
          DeviceNode dn = pm.nodes[g.nodeBegin + q / 2];
          if (outsideLds(q) && (q & 1)) std::memcpy(&dn.value, &dn.meta, sizeof(dn.value));
          return dn;
        };
        auto originAt = [&](uint32_t q) { return q & kTailBit ? pm.tailOrigin[q & ~kTailBit] : pm.nodeOrigin[(size_t)g.nodeBegin * 2 + q]; };
        auto isLeaf = [&](uint32_t q) {
          if (outsideLds(q)) return true;
          const DeviceNode dn = nodeAt(q);
          return q & kTailBit ? (dn.meta >> kTailFeatureBits) == (q & ~kTailBit) : MetaChild(dn.meta) / 4 == q;
        };
        auto leftOf = [&](uint32_t q) -> uint32_t { // the left child (same notation) of a split
          const DeviceNode dn = nodeAt(q);
          if (q & kTailBit) return kTailBit | (dn.meta >> kTailFeatureBits);
          return resolve(MetaChild(dn.meta) / 4);
        };
        auto rightOf = [&](uint32_t q) -> uint32_t {
          const DeviceNode dn = nodeAt(q);
          if (q & kTailBit) return kTailBit | ((dn.meta >> kTailFeatureBits) + 1);
          const uint32_t left = MetaChild(dn.meta) / 4;
          return resolve(left + (left >= g.nodeCount * 2 ? 1 : 2));
        };
        auto featureOf = [&](uint32_t q) -> int32_t {
          const DeviceNode dn = nodeAt(q);
          return q & kTailBit ? (int32_t)(dn.meta & ((1u << kTailFeatureBits) - 1u)) : (int32_t)pm.plan.FeatureOfOffset(MetaFeature(dn.meta));
        };
        Tree tree;
        tree.classId = pm.bundles[bi].classId;
        std::vector<uint32_t> queue{resolve(pm.bundles[bi].root[k] / 4)};
        size_t total = 0;
        for (size_t head = 0; head < queue.size(); ++head) {
          total = std::max<size_t>(total, (size_t)originAt(queue[head]) + 1);
          if (!isLeaf(queue[head])) { queue.push_back(leftOf(queue[head])); queue.push_back(rightOf(queue[head])); }
        }
        tree.value.assign(total, 0.f);
        tree.feature.assign(total, 0);
        tree.left.assign(total, -1);
        tree.right.assign(total, -1);
        for (uint32_t q : queue) {
          const DeviceNode dn = nodeAt(q);
          const int32_t me = originAt(q);
          tree.value[me] = dn.value;
          const bool leaf = isLeaf(q);
          if (!leaf && pm.plan.quantizedRows) { // rank -> threshold through the binning table
            uint32_t j;
            std::memcpy(&j, &dn.value, sizeof(j));
            const int32_t f = featureOf(q);
            const int32_t chunk = pm.binChunkFeatures;
            tree.value[me] = pm.binThresholds[((size_t)(f / chunk) * pm.binTableDepth + j) * chunk + (f % chunk)];
          }
          if (!leaf && pm.plan.rankRows16) {
            uint32_t j;
            std::memcpy(&j, &dn.value, sizeof(j));
            tree.value[me] = pm.rankThresholds.at((size_t)featureOf(q)).at(j);
          }
          if (!leaf) {
            tree.feature[me] = featureOf(q);
            tree.left[me] = originAt(leftOf(q));
            tree.right[me] = originAt(rightOf(q));
          }
        }
        return tree;
      }
  throw Error("tree not found in packed model");
}

} // namespace tbamd
