// The launch plan that is chosen for a forest holds it: ChoosePlan and PackForest over forests at the edges of the forms.
#include "packer.h"
#include "tuner.h"

#include <cstdio>
#include <cstring>

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

int main(int argc, char **argv) {
  const auto asked = [&](const char *name) { return argc < 2 || std::strcmp(argv[1], name) == 0; };
  if (asked("big_trees")) BigTrees();
  if (asked("tail_limit")) TailLimit();
  if (gFailures) return 1;
  std::printf("ok\n");
  return 0;
}
