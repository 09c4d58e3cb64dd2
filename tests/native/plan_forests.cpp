// The launch plan that is chosen for a forest holds it: ChoosePlan and PackForest over forests at the edges of the forms.
#include "packer.h"
#include "tuner.h"

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <limits>

using namespace tbamd;

static int gFailures = 0;
#define EXPECT(cond, ...)                                                                                              \
  do {                                                                                                                 \
    if (!(cond) && ++gFailures < 20) std::printf("FAILED %s: ", #cond), std::printf(__VA_ARGS__), std::printf("\n"); \
  } while (0)

// A tree of `nodes` (odd) nodes, level by level as full as they go.
static Tree FullTree(int32_t nodes, int32_t numFeatures) {
  Tree tree;
  for (int32_t n = 0; n < nodes; ++n) {
    const bool inner = 2 * n + 2 < nodes;
    tree.value.push_back(inner ? 0.25f * (float)(n % 17) : 0.01f * (float)(n % 7));
    tree.feature.push_back(inner ? n % numFeatures : 0);
    tree.left.push_back(inner ? 2 * n + 1 : -1);
    tree.right.push_back(inner ? 2 * n + 2 : -1);
  }
  return tree;
}

// The same with a spine on the left down to `depth`: few of its leaves are on the last level.
static Tree SpinedTree(int32_t nodes, int32_t depth, int32_t numFeatures) {
  Tree tree = FullTree(nodes, numFeatures);
  size_t at = 0;
  int32_t level = 0;
  for (; !tree.IsLeaf((int32_t)at); ++level) at = (size_t)tree.left[at];
  for (; level < depth; ++level) {
    const int32_t child = (int32_t)tree.NumNodes();
    tree.left[at] = child;
    tree.right[at] = child + 1;
    for (int i = 0; i < 2; ++i) {
      tree.value.push_back(0.5f);
      tree.feature.push_back(0);
      tree.left.push_back(-1);
      tree.right.push_back(-1);
    }
    at = (size_t)child;
  }
  return tree;
}

static Forest ForestOf(int32_t numFeatures, int32_t trees, int32_t nodes) {
  Forest forest;
  forest.numFeatures = numFeatures;
  forest.trees.assign((size_t)trees, FullTree(nodes, numFeatures));
  return forest;
}

// One to ten trees up to the largest a tree group can hold, batches around every rule on the number of row blocks.
static void BigTrees() {
  const DeviceLimits limits;
  long packed = 0;
  for (int32_t features = 20; features <= 62; features += 6)
    for (int32_t trees : {1, 2, 3, 10})
      for (int32_t nodes : {2047, 5501, 6401, 7001, 7501, 8001, 8189}) {
        const Forest forest = ForestOf(features, trees, nodes);
        for (int64_t batch : {129, 1000, 32768, 65536, 65537, 131073}) {
          try {
            const PackedModel pm = PackForest(forest, ChoosePlan(forest, batch, nullptr, limits));
            EXPECT(pm.LdsBytes() <= (size_t)limits.ldsBytesPerBlock, "%d features, %d trees of %d nodes, %lld rows: %zu bytes of LDS", features, trees,
                   nodes, (long long)batch, pm.LdsBytes());
            ++packed;
          } catch (const Error &e) {
            EXPECT(false, "%d features, %d trees of %d nodes, %lld rows: %s", features, trees, nodes, (long long)batch, e.what());
          }
        }
      }
  std::printf("big trees: %ld\n", packed);
}

// Deep forests with as many nodes below the cuts as the tail array has places, and with one tree more.
static void TailLimit() {
  const DeviceLimits limits;
  LaunchPlan plan;
  std::vector<int32_t> cuts;
  const struct { int32_t features, nodes; } shapes[] = {{28, 16383}, {28, 21391}, {10, 9665}, {10, 210345}, {200, 9001}};
  for (auto shape : shapes) {
    Forest forest = ForestOf(shape.features, 1, shape.nodes);
    EXPECT(ChooseDeepWalk(forest, limits, &plan, &cuts), "%d features, %d nodes", shape.features, shape.nodes);
    const size_t perTree = PackWithCuts(forest, plan, cuts).tailNodes.size() - 1, most = (kMaxTailNodes - 1) / perTree;
    forest = ForestOf(shape.features, (int32_t)most, shape.nodes);
    EXPECT(ChooseDeepWalk(forest, limits, &plan, &cuts), "%zu trees of %d nodes, %d features", most, shape.nodes, shape.features);
    try {
      const PackedModel pm = PackWithCuts(forest, plan, cuts);
      EXPECT(pm.tailNodes.size() == most * perTree + 1, "%zu trees of %d nodes, %d features: %zu", most, shape.nodes, shape.features, pm.tailNodes.size());
    } catch (const Error &e) {
      EXPECT(false, "%zu trees of %d nodes, %d features: %s", most, shape.nodes, shape.features, e.what());
    }
    forest.trees.push_back(forest.trees[0]);
    EXPECT(!ChooseDeepWalk(forest, limits, &plan, &cuts), "%zu trees of %d nodes, %d features", most + 1, shape.nodes, shape.features);
  }
}

// Nodes that no walk reaches (pruned models keep them) behind those of a tree: they take no place in any form.
static Tree WithUnreachable(Tree tree, int32_t count) {
  tree.value.insert(tree.value.end(), (size_t)count, 3.0f);
  tree.feature.insert(tree.feature.end(), (size_t)count, 0);
  tree.left.insert(tree.left.end(), (size_t)count, -1);
  tree.right.insert(tree.right.end(), (size_t)count, -1);
  return tree;
}

static void UnreachableNodes() {
  const DeviceLimits limits;
  for (int32_t features : {12, 120})
    for (int32_t count : {1, 2, 700, 9000}) {
      Forest forest, whole;
      forest.numFeatures = whole.numFeatures = features;
      for (int32_t nodes : {16383, 8191, 31, 1, 9001, 301}) { // (cut, and small enough to stay whole)
        whole.trees.push_back(FullTree(nodes, features));
        forest.trees.push_back(WithUnreachable(whole.trees.back(), count));
      }
      forest.Validate();
      LaunchPlan plan, planOfWhole;
      std::vector<int32_t> cuts, cutsOfWhole;
      EXPECT(ChooseDeepWalk(forest, limits, &plan, &cuts) && ChooseDeepWalk(whole, limits, &planOfWhole, &cutsOfWhole) && cuts == cutsOfWhole,
             "%d features, %d nodes", features, count);
      try {
        const PackedModel pm = PackWithCuts(forest, plan, cuts), pmOfWhole = PackWithCuts(whole, planOfWhole, cutsOfWhole);
        EXPECT(pm.groups.size() == pmOfWhole.groups.size() && pm.tailNodes.size() == pmOfWhole.tailNodes.size() && pm.treesDeferred == pmOfWhole.treesDeferred,
               "%d features, %d nodes: %zu groups and %zu tail nodes, %zu and %zu without", features, count, pm.groups.size(), pm.tailNodes.size(),
               pmOfWhole.groups.size(), pmOfWhole.tailNodes.size());
        for (size_t t = 0; t < whole.trees.size(); ++t) {
          const Tree tree = UnpackTree(pm, (int32_t)t);
          EXPECT(tree.value == whole.trees[t].value && tree.left == whole.trees[t].left && tree.right == whole.trees[t].right, "%d features, %d nodes, tree %zu",
                 features, count, t);
        }
      } catch (const Error &e) {
        EXPECT(false, "%d features, %d nodes: %s", features, count, e.what());
      }
      // deferred tails by a profile, of a tree that a tree group holds and that all rows leave at its first leaf
      Tree tree{{0.5f, 0.1f}, {0, 0}, {1, -1}, {2, -1}, 0};
      const Tree rest = FullTree(2047, features);
      for (size_t n = 0; n < rest.NumNodes(); ++n) {
        tree.value.push_back(rest.value[n]);
        tree.feature.push_back(rest.feature[n]);
        tree.left.push_back(rest.left[n] < 0 ? -1 : rest.left[n] + 2);
        tree.right.push_back(rest.right[n] < 0 ? -1 : rest.right[n] + 2);
      }
      forest.trees = {WithUnreachable(tree, count % 2000)};
      HitCountProfile profile;
      profile.numRows = 100;
      profile.hits.assign(1, std::vector<int64_t>(forest.trees[0].NumNodes(), 0));
      profile.hits[0][0] = profile.hits[0][1] = 100;
      WalkOptions walk;
      walk.peelWalks = true;
      try {
        const LaunchPlan peeled = ChoosePlan(forest, 100000, nullptr, limits, walk);
        EXPECT(peeled.deferTails, "%d features, %d nodes", features, count);
        EXPECT(PackForest(forest, peeled, &profile).treesDeferred == 1, "%d features, %d nodes", features, count);
      } catch (const Error &e) {
        EXPECT(false, "%d features, %d nodes, by a profile: %s", features, count, e.what());
      }
    }
}

// Splits that no walk reaches may name any feature and compare with anything: they are no thresholds of the rows' ranks.
static void UnreachableSplits() {
  const DeviceLimits limits;
  for (int32_t features : {12, 700}) {
    Forest forest = ForestOf(features, 3, 255);
    const int32_t most = MaxThresholdsPerFeature(forest);
    for (Tree &tree : forest.trees)
      for (int32_t n = 0; n < 400; ++n) {
        tree.value.push_back(n % 3 ? 1000.0f + (float)n : std::numeric_limits<float>::quiet_NaN());
        tree.feature.push_back(n % 2 ? 0 : 1 << 24);
        tree.left.push_back(1);
        tree.right.push_back(2);
      }
    forest.Validate();
    EXPECT(MaxThresholdsPerFeature(forest) == most, "%d features: %d and %d", features, (int)MaxThresholdsPerFeature(forest), (int)most);
    for (int64_t batch : {1, 1000, 1 << 20}) {
      LaunchPlan plan = ChoosePlan(forest, batch, nullptr, limits);
      (void)PackForest(forest, plan);
      if (features > 100 || plan.kernel != LaunchPlan::Kernel::kRowParallelLds) continue;
      plan.rankRows16 = true;
      (void)PackForest(forest, plan);
    }
    (void)PackRankStream(forest);
    (void)PackFewRows(forest);
  }
}

// Small forests with peeled walks: no deferred tails in the blocks of their own, in others as before; one tree group either way.
static void SmallPeeled() {
  const DeviceLimits limits;
  WalkOptions walk;
  walk.peelWalks = true;
  for (int32_t features : {5, 20, 30})
    for (int32_t nodes : {31, 127, 1023, 2047}) {
      const Forest forest = ForestOf(features, std::max(1, 2900 / nodes), nodes);
      HitCountProfile profile;
      profile.numRows = 1;
      for (const Tree &tree : forest.trees) profile.hits.emplace_back(tree.NumNodes(), 1);
      for (int64_t batch : {20000, 60000, 100000, 200000, 1 << 20}) {
        for (bool later : {false, true}) { // (with the model, or asked for when the runner is there)
          LaunchPlan plan = ChoosePlan(forest, batch, nullptr, limits, later ? WalkOptions() : walk);
          if (later) plan.peelWalks = true, plan.deferTails = DeferTailsFit(forest, &plan);
          EXPECT((plan.rowsPerBlock == 128 && plan.treeThreads == 4) == (batch != 100000), "%lld rows: %d x %d", (long long)batch, plan.rowsPerBlock,
                 plan.treeThreads);
          EXPECT(plan.deferTails == (batch == 100000) && plan.peelWalks, "%d features, %zu trees of %d nodes, %lld rows: %d x %d, groups of %d bytes", features, forest.trees.size(), nodes,
                 (long long)batch, plan.rowsPerBlock, plan.treeThreads, plan.groupBytes);
          const PackedModel pm = PackForest(forest, plan, &profile);
          EXPECT(pm.groups.size() == 1 && pm.LdsBytes() <= (size_t)limits.ldsBytesPerBlock / 2, "%d features, %zu trees of %d nodes, %lld rows: %zu groups",
                 features, forest.trees.size(), nodes, (long long)batch, pm.groups.size());
        }
      }
    }
}

// The block shapes of batches of up to a block of 256 rows for each compute unit, and of small forests, either side of their rules' lines.
static void SmallBatches() {
  const DeviceLimits limits;
  const struct { int64_t batch; int32_t trees, nodes, features, rows, threads; } shapes[] = {
      {32768, 30, 255, 20, 128, 8},  {32769, 30, 255, 20, 256, 4},                                // half of the units have a block, and more
      {40000, 77, 63, 20, 256, 4},   {40000, 78, 63, 20, 128, 8},                                 // 385 and 390 levels, one group
      {40000, 107, 127, 20, 256, 4}, {40000, 108, 127, 20, 128, 8},                               // 642 and 648, two groups
      {40000, 73, 63, 50, 256, 4},   {40000, 74, 63, 50, 128, 8},                                 // 365 and 370, two groups beside 256 rows and one beside 128
      {65536, 100, 255, 20, 128, 8}, {65537, 100, 255, 20, 256, 4},                               // four groups
      {131072, 59, 31, 50, 256, 4},  {131073, 59, 31, 50, 128, 4},                                // a round of blocks of 256 rows, and more
      {300000, 59, 31, 50, 128, 4},  {300000, 60, 31, 50, 256, 4},                                // four fit a unit's LDS, and three
      {163840, 60, 31, 50, 128, 4},  {163841, 60, 31, 50, 256, 4}};                               // three, of a round and a quarter
  for (auto s : shapes) {
    const Forest forest = ForestOf(s.features, s.trees, s.nodes);
    const LaunchPlan plan = ChoosePlan(forest, s.batch, nullptr, limits);
    EXPECT(plan.treeSlices > 1 || (plan.rowsPerBlock == s.rows && plan.treeThreads == s.threads), "%lld rows, %d trees of %d nodes: %d x %d",
           (long long)s.batch, s.trees, s.nodes, plan.rowsPerBlock, plan.treeThreads);
    EXPECT(plan.treeSlices == 1, "%lld rows, %d trees of %d nodes: %d slices", (long long)s.batch, s.trees, s.nodes, plan.treeSlices);
  }
}

// Classifiers walk two trees side by side for classes of the tree threads' own only where they are packed so, or where groups hold
// few trees.
static void TwoTreesOfClasses() {
  const DeviceLimits limits;
  long own = 0, few = 0;
  for (int32_t features : {12, 33, 54, 78, 113})
    for (int32_t classes : {3, 5, 7, 10, 13, 16})
      for (int32_t trees : {61, 160, 321, 607}) {
        Forest forest = ForestOf(features, trees, trees % 2 ? 127 : 255);
        forest.numClasses = classes;
        for (int32_t t = 0; t < trees; ++t) forest.trees[(size_t)t].classId = t % classes;
        for (int64_t batch : {2600, 30000, 190000}) {
          const LaunchPlan plan = ChoosePlan(forest, batch, nullptr, limits);
          if (plan.interleave != 2 || plan.kernel != LaunchPlan::Kernel::kRowParallelLds) continue;
          const double held = (double)plan.groupBytes / (double)(forest.trees[0].NumNodes() * kNodeBytes);
          if (held < std::min(24.0, 2.4 * plan.treeThreads + 3.4)) {
            ++few;
            continue;
          }
          ++own;
          EXPECT(PacksOwnClasses(forest, plan) && PackForest(forest, plan).ownClasses, "%d features, %d classes, %d trees, %lld rows: groups of %.1f trees",
                 features, classes, trees, (long long)batch, held);
        }
      }
  EXPECT(own > 0 && few > 0, "%ld, %ld", own, few);
}

// Two trees side by side give no slice half as many groups again as four do; the planner counts the groups that are packed.
static void TwoTreesOfSlices() {
  const DeviceLimits limits;
  long two = 0, kept = 0;
  for (int32_t features : {8, 26, 33, 57, 90, 130})
    for (int32_t trees : {61, 80, 89, 161, 300})
      for (int32_t nodes : {127, 255, 511})
        for (int64_t batch : {4000, 7414, 12708, 16925, 30000}) {
          Forest forest = ForestOf(features, trees, nodes);
          for (size_t t = 0; t < forest.trees.size(); t += 3) forest.trees[t] = FullTree(nodes / 4 * 2 + 1, features);
          LaunchPlan plan = ChoosePlan(forest, batch, nullptr, limits);
          if (plan.kernel != LaunchPlan::Kernel::kRowParallelLds || plan.treeSlices == 1) continue;
          const bool chosen = plan.interleave == 2;
          size_t turns[2];
          for (int32_t k : {2, 4}) {
            plan.interleave = k;
            const size_t groups = PackForest(forest, plan).groups.size();
            EXPECT(groups == (size_t)CountTreeGroups(forest, plan), "%d features, %d trees of %d nodes, %lld rows: %zu and %d groups", features, trees, nodes,
                   (long long)batch, groups, CountTreeGroups(forest, plan));
            turns[k / 4] = (groups + (size_t)plan.treeSlices - 1) / (size_t)plan.treeSlices;
          }
          EXPECT(!chosen || turns[0] * 2 < turns[1] * 3, "%d features, %d trees of %d nodes, %lld rows: %zu and %zu groups a slice", features, trees, nodes,
                 (long long)batch, turns[0], turns[1]);
          ++(chosen ? two : kept);
        }
  EXPECT(two > 0 && kept > 0, "%ld, %ld", two, kept);
}

// Peeled walks that end in no deferred tails (classes, rows of word offsets, no room for the queues) are laid out as others are, and
// so planned; those with deferred tails keep all leaves in LDS, and the slices' turns are counted that way.
static void PlansOfPeeledWalks() {
  const DeviceLimits limits;
  WalkOptions walk;
  walk.peelWalks = true;
  long whole = 0, tails = 0, outside = 0, two = 0;
  for (int32_t features : {8, 33, 57, 130, 300})
    for (int32_t classes : {0, 3})
      for (int32_t trees : {61, 89, 161})
        for (int32_t nodes : {127, 511})
          for (int64_t batch : {7414, 12708, 30000, 262144}) {
            Forest forest = ForestOf(features, trees, nodes);
            forest.numClasses = classes;
            for (int32_t t = 0; t < trees; ++t) {
              if (t % 3 == 0) forest.trees[(size_t)t] = FullTree(nodes / 4 * 2 + 1, features);
              forest.trees[(size_t)t].classId = classes ? t % classes : 0;
            }
            const LaunchPlan plain = ChoosePlan(forest, batch, nullptr, limits), peeled = ChoosePlan(forest, batch, nullptr, limits, walk);
            if (plain.kernel != LaunchPlan::Kernel::kRowParallelLds || plain.quantizedRows) continue;
            if (!peeled.deferTails) {
              ++whole;
              outside += PackForest(forest, plain).leavesOutside;
              EXPECT(peeled.interleave == plain.interleave && peeled.groupBytes == plain.groupBytes && peeled.treeSlices == plain.treeSlices,
                     "%d features, %d classes, %d trees of %d nodes, %lld rows: %d and %d trees a lane", features, classes, trees, nodes, (long long)batch,
                     plain.interleave, peeled.interleave);
            } else if (peeled.treeSlices > 1 && peeled.interleave == 2) {
              ++two;
              LaunchPlan p = peeled; // (as it was when the trees a lane were chosen: no room given to the queues yet)
              p.groupBytes = plain.groupBytes;
              int64_t turns[2];
              for (int32_t k : {2, 4}) {
                p.interleave = k;
                turns[k / 4] = (CountTreeGroups(forest, p) + p.treeSlices - 1) / p.treeSlices;
              }
              EXPECT(turns[0] * 2 < turns[1] * 3, "%d features, %d trees of %d nodes, %lld rows: %lld and %lld groups a slice", features, trees, nodes,
                     (long long)batch, (long long)turns[0], (long long)turns[1]);
            }
            tails += peeled.deferTails;
          }
  EXPECT(whole > 0 && tails > 0 && outside > 0 && two > 0, "%ld, %ld, %ld, %ld", whole, tails, outside, two);
}

// Numbers of features that files can hold: too many for any row in LDS, and the last ones that can be counted.
static void MostFeatures() {
  const DeviceLimits limits;
  const int32_t last = std::numeric_limits<int32_t>::max();
  for (int32_t features : {16384, 65536, 1 << 24, last - 3, last - 2, last - 1, last}) {
    Forest forest = ForestOf(100, 4, 63);
    forest.numFeatures = features;
    bool valid = true;
    try {
      forest.Validate();
    } catch (const Error &) {
      valid = false;
    }
    EXPECT(valid == (features <= last - 2), "%d features", features);
    if (!valid) continue;
    for (int64_t batch : {1, 1000, 1 << 20}) {
      const LaunchPlan plan = ChoosePlan(forest, batch, nullptr, limits);
      EXPECT(plan.kernel == LaunchPlan::Kernel::kGlobalWalk && PackForest(forest, plan).globalTrees.size() == 4, "%d features, %lld rows", features, (long long)batch);
    }
  }
}

// Classifiers under every order that a profile gives their trees: what the planner took to be the tree threads' own classes may meet
// after all, and then finds its room, two blocks to a compute unit where the plan was made for two.
static void RoomOfOwnClasses() {
  const DeviceLimits limits;
  uint64_t state = 1;
  const auto pick = [&](int32_t low, int32_t high) {
    state = state * 6364136223846793005ull + 1442695040888963407ull;
    return low + (int32_t)((state >> 33) % (uint64_t)(high - low + 1));
  };
  long roomy = 0, meet = 0;
  for (int32_t i = 0; i < 800; ++i) {
    const bool wide = i % 2; // (one block per compute unit, and two)
    const bool spined = i % 4 / 2; // (all leaves of these stay in LDS)
    const int32_t features = wide ? pick(380, 520) : pick(20, 110), classes = wide ? pick(10, 16) : pick(3, 9), trees = pick(40, 110);
    Forest forest = ForestOf(features, trees, 3);
    forest.numClasses = classes;
    HitCountProfile profile;
    profile.numRows = 1000;
    const int32_t biggest = wide ? pick(190, 255) : pick(330, 511);
    for (int32_t t = 0; t < trees; ++t) { // of one depth and many sizes, which the profile brings into order
      const int32_t nodes = pick(spined ? biggest / 3 : wide ? 131 : 257, biggest) / 2 * 2 + 1;
      Tree &tree = forest.trees[(size_t)t] = spined ? SpinedTree(nodes, 12, features) : FullTree(nodes, features);
      tree.classId = t % classes;
      std::vector<int64_t> hits(tree.NumNodes(), 0);
      hits[0] = profile.numRows;
      const bool big = (int32_t)tree.NumNodes() * 4 > biggest * 3;
      for (size_t n = 0; n < tree.NumNodes(); ++n)
        if (!tree.IsLeaf((int32_t)n)) {
          hits[(size_t)tree.left[n]] = big ? 0 : hits[n]; // (the deeper side)
          hits[(size_t)tree.right[n]] = big ? hits[n] : 0;
        }
      profile.hits.push_back(hits);
    }
    const int64_t batch = pick(2000, 600000);
    WalkOptions walk;
    walk.peelWalks = true;
    LaunchPlan later = ChoosePlan(forest, batch, nullptr, limits);
    const PackedModel plain = PackForest(forest, later);
    later.peelWalks = true; // (asked for when the runner is there)
    for (const LaunchPlan &plan : {ChoosePlan(forest, batch, nullptr, limits, walk), later}) {
      if (plan.kernel != LaunchPlan::Kernel::kRowParallelLds || plan.quantizedRows) continue;
      const PackedModel pm = PackForest(forest, plan, &profile);
      EXPECT(pm.LdsBytes() <= (size_t)limits.ldsBytesPerBlock && (plain.LdsBytes() * 2 > (size_t)limits.ldsBytesPerBlock || pm.LdsBytes() * 2 <= (size_t)limits.ldsBytesPerBlock),
             "%d features, %d classes, %d trees, %lld rows: %zu and %zu bytes of LDS, own classes %d and %d", features, classes, trees, (long long)batch,
             plain.LdsBytes(), pm.LdsBytes(), plain.ownClasses, pm.ownClasses);
      if (plain.ownClasses && plan.ownGroupBytes > 0 && plain.groupBytes == plan.ownGroupBytes) ++(pm.ownClasses ? roomy : meet);
    }
  }
  EXPECT(roomy > 0 && meet > 0, "%ld, %ld", roomy, meet);
}

int main(int argc, char **argv) {
  const auto asked = [&](const char *name) { return argc < 2 || std::strcmp(argv[1], name) == 0; };
  if (asked("big_trees")) BigTrees();
  if (asked("tail_limit")) TailLimit();
  if (asked("unreachable_nodes")) UnreachableNodes();
  if (asked("unreachable_splits")) UnreachableSplits();
  if (asked("small_peeled")) SmallPeeled();
  if (asked("small_batches")) SmallBatches();
  if (asked("two_trees_of_classes")) TwoTreesOfClasses();
  if (asked("two_trees_of_slices")) TwoTreesOfSlices();
  if (asked("most_features")) MostFeatures();
  if (asked("room_of_own_classes")) RoomOfOwnClasses();
  if (asked("plans_of_peeled_walks")) PlansOfPeeledWalks();
  if (gFailures) return 1;
  std::printf("ok\n");
  return 0;
}
