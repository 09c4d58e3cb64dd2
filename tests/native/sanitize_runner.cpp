// Drives the C ABI (runtime.cpp + runner.cpp + the host sources) over the host-only HIP stand-in
// (hip_host_shim.cpp) so that AddressSanitizer / UBSan / ThreadSanitizer see every buffer the runner
// sizes and every copy it makes: host entry points with pageable and "pinned" inputs of many sizes (one
// copy, staged pieces, windows), device entry points, plan changes, the plan search, the compiled-model
// file, the entry points on a caller's stream.  Predictions are compared with a plain walk of the forest.
#include "../../include/tbruntime_amd.h"

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstdint>
#include <cstring>
#include <fstream>
#include <iterator>
#include <random>
#include <string>
#include <vector>

extern "C" long shimFewRows, shimSplits, shimStreams, shimDeferred, shimLaunchesToGo, shimNoLaunches; // hip_host_shim.cpp
extern "C" int shimBusyStreams(hipStream_t except);

namespace {

struct HostTree {
  std::vector<float> value;
  std::vector<int32_t> feature, left, right;
  int32_t classId = 0;
};

struct HostForest {
  std::vector<HostTree> trees;
  int64_t numFeatures = 0, numClasses = 0, transform = 0;
  double initial = 0.0;
};

int gFailures = 0;
#define EXPECT(cond, ...)                                                                                              \
  do {                                                                                                                 \
    if (!(cond)) {                                                                                                     \
      std::printf("FAILED %s:%d: ", __FILE__, __LINE__);                                                               \
      std::printf(__VA_ARGS__);                                                                                        \
      std::printf(" [%s]\n", tbmi_last_error());                                                                       \
      ++gFailures;                                                                                                     \
    }                                                                                                                  \
  } while (0)

HostForest LoadForest(const char *path) {
  HostForest f;
  const intptr_t h = tbmi_load_forest(path, "xgboost_json", 0);
  if (!h) {
    std::printf("cannot load %s: %s\n", path, tbmi_last_error());
    std::exit(2);
  }
  int64_t info[6];
  tbmi_forest_info(h, info, &f.initial);
  f.numFeatures = info[1];
  f.numClasses = info[2];
  f.transform = info[3];
  f.trees.resize((size_t)info[0]);
  for (size_t t = 0; t < f.trees.size(); ++t) {
    const int32_t n = tbmi_forest_tree_size(h, (int32_t)t);
    HostTree &tree = f.trees[t];
    tree.value.resize(n);
    tree.feature.resize(n);
    tree.left.resize(n);
    tree.right.resize(n);
    tbmi_forest_tree(h, (int32_t)t, tree.value.data(), tree.feature.data(), tree.left.data(), tree.right.data(), &tree.classId);
  }
  tbmi_delete_forest(h);
  return f;
}

// Prediction of one row as RunInference returns it (class id for classifiers).
float Predict(const HostForest &f, const float *row, int32_t *leafIds) {
  std::vector<double> sums((size_t)std::max<int64_t>(1, f.numClasses), 0.0);
  for (size_t t = 0; t < f.trees.size(); ++t) {
    const HostTree &tree = f.trees[t];
    int32_t n = 0;
    while (tree.left[n] != -1) n = row[tree.feature[n]] < tree.value[n] ? tree.left[n] : tree.right[n];
    if (leafIds) leafIds[t] = n;
    sums[f.numClasses > 0 ? tree.classId : 0] += (double)tree.value[n];
  }
  if (f.numClasses == 0) {
    const double margin = f.initial + sums[0];
    return (float)(f.transform == 1 ? 1.0 / (1.0 + std::exp(-margin)) : margin);
  }
  float best = -INFINITY;
  int bestClass = 0;
  for (int c = 0; c < (int)f.numClasses; ++c) {
    const float m = (float)(f.initial + sums[c]);
    if (!(best > m)) best = m, bestClass = c;
  }
  return (float)bestClass;
}

bool Close(float a, float b) { return std::fabs((double)a - (double)b) <= 1e-6 + 1e-5 * std::fabs((double)b); }

struct Case {
  HostForest forest;
  std::string path;
  std::vector<float> x;        // rows x F
  std::vector<float> expected; // rows
  int64_t rows = 0;
};

void Compare(const Case &c, const float *got, int64_t first, int64_t rows, const char *what, hipStream_t mine = nullptr) {
  EXPECT(shimBusyStreams(mine) == 0, "%s returned with work under way", what);
  int64_t bad = 0;
  for (int64_t r = 0; r < rows; ++r) bad += !Close(got[r], c.expected[first + r]);
  EXPECT(bad == 0, "%s: %lld of %lld rows differ (%s)", what, (long long)bad, (long long)rows, c.path.c_str());
}

// Leaf hit counts of the case's own rows in the reference's profile format (first line `numTrees, numRows`,
// then per tree `hitCount, depth` for every leaf in node order).
std::string WriteProfile(const Case &c, const std::string &path) {
  const int64_t F = c.forest.numFeatures;
  const size_t T = c.forest.trees.size();
  std::vector<std::vector<int64_t>> hits(T);
  for (size_t t = 0; t < T; ++t) hits[t].assign(c.forest.trees[t].value.size(), 0);
  std::vector<int32_t> ids(T);
  for (int64_t r = 0; r < c.rows; ++r) {
    Predict(c.forest, c.x.data() + r * F, ids.data());
    for (size_t t = 0; t < T; ++t) ++hits[t][ids[t]];
  }
  FILE *out = std::fopen(path.c_str(), "w");
  std::fprintf(out, "%zu, %lld\n", T, (long long)c.rows);
  for (size_t t = 0; t < T; ++t) {
    const HostTree &tree = c.forest.trees[t];
    bool first = true;
    for (size_t n = 0; n < tree.value.size(); ++n) {
      if (tree.left[n] != -1) continue;
      std::fprintf(out, "%s%lld, 0", first ? "" : ", ", (long long)hits[t][n]);
      first = false;
    }
    std::fprintf(out, "\n");
  }
  std::fclose(out);
  return path;
}

intptr_t MakeRunner(const Case &c, int32_t batch, bool int8Classes, int32_t tileSize = 1, int32_t tilingType = 0,
                    const char *profile = "") {
  const intptr_t options = CreateCompilerOptions();
  Set_batchSize(options, batch);
  Set_tileSize(options, tileSize);
  Set_tilingType(options, tilingType);
  Set_statsProfileCSVPath(options, profile);
  if (int8Classes) {
    Set_returnTypeWidth(options, 8);
    Set_returnTypeFloatType(options, 0);
  }
  const intptr_t runner = CreateInferenceRunner(c.path.c_str(), "", options);
  DeleteCompilerOptions(options);
  EXPECT(runner != 0 || tileSize > 1, "CreateInferenceRunner");
  return runner;
}

std::string Describe(intptr_t runner) {
  char text[1024];
  tbmi_describe_plan(runner, text, sizeof(text));
  return text;
}

// The kernels of the runner's own launch plan, whatever forms take its calls otherwise (batches of a few rows, streamed
// bundles): the plan the description names, pinned.
void PinOwnPlan(intptr_t runner) {
  char text[1024];
  tbmi_describe_plan(runner, text, sizeof(text));
  const auto field = [&](const char *name) {
    const char *at = std::strstr(text, (std::string(" ") + name + "=").c_str());
    return at ? std::atoi(at + std::strlen(name) + 2) : 0;
  };
  const int32_t rows = field("rowsPerBlock"), k = field("interleave"), bytes = field("groupBytes"), slices = field("treeSlices");
  int32_t rc;
  if (std::strstr(text, "kernel=tree_parallel")) rc = tbmi_set_tree_parallel_plan(runner, rows, field("treeLanes"), k, bytes, slices);
  else if (std::strstr(text, "kernel=global_walk")) rc = tbmi_set_global_walk_plan(runner, rows, k, slices);
  else if (field("quantizedRows")) rc = tbmi_set_quantized_plan(runner, field("treeThreads"), k, bytes, slices);
  else if (field("rankRows16")) rc = tbmi_set_rank16_plan(runner, rows, field("treeThreads"), k, bytes, slices);
  else rc = tbmi_set_plan(runner, rows, field("treeThreads"), k, bytes, slices);
  EXPECT(rc == 0, "pinning %s", text);
}

// SANITIZE_QUICK=1: only the largest batch through the host entry points and the default plan through the
// device entry points (the thread sanitizer's slower build looks at the copier threads, not at plan shapes).
bool Quick() { return std::getenv("SANITIZE_QUICK") != nullptr; }

void HostEntryPoints(const Case &c, bool pinned = false) {
  const int64_t F = c.forest.numFeatures;
  // exact-size result buffers (heap, so that an overrun is seen), several batch sizes incl. the staged path
  for (int64_t rows : {(int64_t)1, (int64_t)63, (int64_t)1000, (int64_t)8192, c.rows}) {
    if (rows > c.rows || (Quick() && rows != c.rows)) continue;
    const intptr_t runner = MakeRunner(c, (int32_t)rows, false);
    if (!runner) continue;
    if (pinned) PinOwnPlan(runner);
    std::vector<float> in(c.x.begin(), c.x.begin() + rows * F), out((size_t)rows, -1.f);
    RunInference(runner, in.data(), out.data());
    Compare(c, out.data(), 0, rows, "RunInference");
    RunInference(runner, in.data(), out.data()); // buffers reused
    Compare(c, out.data(), 0, rows, "RunInference again");
    // "pinned" input: memory the runtime knows as host memory is read where it lies
    void *locked = nullptr;
    if (hipHostMalloc(&locked, (size_t)rows * F * sizeof(float), 0) == hipSuccess) {
      std::memcpy(locked, in.data(), (size_t)rows * F * sizeof(float));
      std::fill(out.begin(), out.end(), -1.f);
      RunInference(runner, locked, out.data());
      Compare(c, out.data(), 0, rows, "RunInference pinned");
      (void)hipHostFree(locked);
    }
    // any number of rows through a runner compiled for `rows`
    for (int64_t n : {(int64_t)0, rows / 3, rows, std::min(c.rows, rows * 2 + 5), c.rows}) {
      if (Quick() && n != c.rows) continue;
      std::vector<float> in2(c.x.begin(), c.x.begin() + n * F), out2((size_t)n, -1.f);
      EXPECT(tbmi_run_host(runner, in2.data(), out2.data(), n) == 0, "tbmi_run_host %lld", (long long)n);
      Compare(c, out2.data(), 0, n, "tbmi_run_host");
    }
    const int64_t whole = c.rows / rows * rows;
    if (whole > 0 && whole <= (int64_t)1 << 30 && !Quick()) {
      std::vector<float> in3(c.x.begin(), c.x.begin() + whole * F), out3((size_t)whole, -1.f);
      RunInferenceOnMultipleBatches(runner, in3.data(), out3.data(), (int32_t)whole);
      Compare(c, out3.data(), 0, whole, "RunInferenceOnMultipleBatches");
    }
    DeleteInferenceRunner(runner);
  }
}

// Ids, sums and softmax of a classifier, together and one alone.
void MulticlassOutputs(const Case &c, intptr_t runner, const float *dx, int64_t rows) {
  if (c.forest.numClasses == 0) return;
  const size_t values = (size_t)rows * (size_t)c.forest.numClasses;
  int8_t *cls = nullptr;
  float *margins = nullptr, *probs = nullptr;
  EXPECT(hipMalloc((void **)&cls, (size_t)rows) == hipSuccess, "hipMalloc");
  EXPECT(hipMalloc((void **)&margins, values * sizeof(float)) == hipSuccess, "hipMalloc");
  EXPECT(hipMalloc((void **)&probs, values * sizeof(float)) == hipSuccess, "hipMalloc");
  std::fill_n(margins, values, std::nanf(""));
  std::fill_n(probs, values, std::nanf(""));
  EXPECT(tbmi_run_device_multiclass(runner, dx, rows, cls, margins, probs) == 0, "tbmi_run_device_multiclass");
  for (int64_t r = 0; r < rows; ++r) {
    EXPECT((float)cls[r] == c.expected[r], "class id of row %lld", (long long)r);
    double z = 0.0;
    for (int64_t i = 0; i < c.forest.numClasses; ++i) z += probs[r * c.forest.numClasses + i];
    EXPECT(std::fabs(z - 1.0) < 1e-5, "probabilities of row %lld", (long long)r);
    EXPECT(margins[r * c.forest.numClasses + cls[r]] == *std::max_element(margins + r * c.forest.numClasses, margins + (r + 1) * c.forest.numClasses),
           "sums of row %lld", (long long)r);
  }
  EXPECT(tbmi_run_device_multiclass(runner, dx, rows, nullptr, margins, nullptr) == 0, "tbmi_run_device_multiclass");
  (void)hipFree(cls);
  (void)hipFree(margins);
  (void)hipFree(probs);
}

void DeviceEntryPoints(const Case &c, int64_t rows, int32_t tileSize = 1, int32_t tilingType = 0, const char *profile = "",
                       bool peel = false) {
  const int64_t F = c.forest.numFeatures;
  const int32_t T = (int32_t)c.forest.trees.size();
  const bool multiclass = c.forest.numClasses > 0;
  SetPeeledCodeGenForProbabilityBasedTiling(peel ? 1 : 0);
  const intptr_t runner = MakeRunner(c, (int32_t)rows, multiclass, tileSize, tilingType, profile);
  SetPeeledCodeGenForProbabilityBasedTiling(0);
  if (!runner) {
    // tiled walks are refused where the row tile cannot hold byte offsets (very wide rows), never silently dropped
    EXPECT(tileSize > 1 && std::strstr(tbmi_last_error(), "tile size"), "runner with tile size %d", tileSize);
    return;
  }
  {
    char plan[1024];
    tbmi_describe_plan(runner, plan, sizeof(plan));
    char want[64];
    std::snprintf(want, sizeof(want), " tileSize=%d ", tileSize);
    EXPECT(std::strstr(plan, want) != nullptr, "plan does not carry the tile size: %s", plan);
  }
  float *dx = nullptr;
  void *dout = nullptr;
  int32_t *dids = nullptr;
  EXPECT(hipMalloc((void **)&dx, (size_t)rows * F * sizeof(float)) == hipSuccess, "hipMalloc");
  EXPECT(hipMalloc(&dout, (size_t)rows * tbmi_result_bytes(runner)) == hipSuccess, "hipMalloc");
  EXPECT(hipMalloc((void **)&dids, (size_t)rows * T * sizeof(int32_t)) == hipSuccess, "hipMalloc");
  std::memcpy(dx, c.x.data(), (size_t)rows * F * sizeof(float));
  std::vector<int32_t> wantIds((size_t)rows * T);
  for (int64_t r = 0; r < rows; ++r) Predict(c.forest, c.x.data() + r * F, wantIds.data() + r * T);

  auto check = [&](const char *what) {
    std::vector<float> got((size_t)rows);
    for (int64_t r = 0; r < rows; ++r)
      got[r] = multiclass ? (float)static_cast<int8_t *>(dout)[r] : static_cast<float *>(dout)[r];
    Compare(c, got.data(), 0, rows, what);
    std::memset(dout, 0x5A, (size_t)rows * tbmi_result_bytes(runner));
  };
  auto runAll = [&](const char *what) {
    EXPECT(tbmi_run_device(runner, dx, dout, rows) == 0, "tbmi_run_device (%s)", what);
    check(what);
    EXPECT(tbmi_run_device_async(runner, dx, dout, rows, nullptr) == 0, "tbmi_run_device_async (%s)", what);
    check(what);
    if (tbmi_run_device_noalloc(runner, dx, dout, rows, nullptr) == 0) check(what);
    else EXPECT(std::strstr(tbmi_last_error(), "scratch memory") != nullptr, "tbmi_run_device_noalloc (%s)", what);
    EXPECT(tbmi_run_device_noalloc(runner, dx, dout, rows / 2, nullptr) == 0 || std::strstr(tbmi_last_error(), "scratch memory"),
           "tbmi_run_device_noalloc half (%s)", what);
    std::memset(dids, 0xFF, (size_t)rows * T * sizeof(int32_t));
    EXPECT(tbmi_dump_leaf_ids(runner, dx, dids, rows) == 0, "tbmi_dump_leaf_ids (%s)", what);
    EXPECT(std::memcmp(dids, wantIds.data(), wantIds.size() * sizeof(int32_t)) == 0, "leaf ids differ (%s)", what);
    double w = 0, f = 0, b = 0;
    EXPECT(tbmi_time_kernels(runner, dx, dout, rows, 2, &w, &f, &b) == 0, "tbmi_time_kernels (%s)", what);
    char small[16], big[1024];
    EXPECT(tbmi_describe_plan(runner, small, sizeof(small)) > 0 && std::strlen(small) == sizeof(small) - 1, "describe (small)");
    EXPECT(tbmi_describe_plan(runner, big, sizeof(big)) > 0, "describe");
  };
  runAll("default plan");
  MulticlassOutputs(c, runner, dx, rows);
  if (tileSize == 1 && tilingType == 0) {
    PinOwnPlan(runner);
    runAll("default plan, pinned");
  }
  if (tileSize > 1) { // block shapes of the tiled walk, the plan search, save and reload
    const int tiledPlans[][5] = {{64, 1, 1, 16384, 1}, {128, 8, 2, 32768, 3}, {256, 4, 4, 40960, 2}, {64, 16, 2, 24576, 5}, {128, 4, 1, 65536, 2}};
    for (auto &p : tiledPlans)
      if (tbmi_set_plan(runner, p[0], p[1], p[2], p[3], p[4]) == 0) runAll("tiled plan");
    EXPECT(tbmi_set_tree_parallel_plan(runner, 4, 64, 1, 0, 1) == -1, "tree-parallel plan must refuse tiles");
    EXPECT(tbmi_set_global_walk_plan(runner, 256, 4, 1) == -1, "global-walk plan must refuse tiles");
    EXPECT(tbmi_set_quantized_plan(runner, 8, 4, 0, 1) == -1, "one-byte rank plan must refuse tiles");
    EXPECT(tbmi_set_rank16_plan(runner, 64, 4, 4, 0, 1) == -1, "two-byte rank plan must refuse tiles");
    if ((F + 1) * 512 * 4 > 0x10000) EXPECT(tbmi_set_plan(runner, 512, 2, 2, 0, 1) == -1, "a row tile of 64 KB must refuse tiles");
    double best = 0;
    EXPECT(tbmi_autotune(runner, dx, rows < 96 ? rows : 96, &best) == 0, "tbmi_autotune (tiled)"); // (a few rows: the search re-packs and launches hundreds of times)
    runAll("tiled, after the plan search");
    const std::string file = std::string(std::getenv("TMPDIR") ? std::getenv("TMPDIR") : "/tmp") + "/sanitize_tiled.tbamd";
    EXPECT(tbmi_save_compiled_model(runner, file.c_str()) == 0, "tbmi_save_compiled_model (tiled)");
    const intptr_t again = tbmi_load_compiled_model(file.c_str(), 0);
    EXPECT(again != 0, "tbmi_load_compiled_model (tiled)");
    if (again) {
      char a[1024], b[1024];
      tbmi_describe_plan(runner, a, sizeof(a));
      tbmi_describe_plan(again, b, sizeof(b));
      EXPECT(std::strcmp(a, b) == 0, "reloaded tiled plan differs: %s / %s", a, b);
      EXPECT(tbmi_run_device(again, dx, dout, rows) == 0, "reloaded tiled runner");
      check("reloaded tiled runner");
      DeleteInferenceRunner(again);
    }
  }
  if (Quick() || tileSize > 1) {
    DeleteInferenceRunner(runner);
    (void)hipFree(dx);
    (void)hipFree(dout);
    (void)hipFree(dids);
    return;
  }
  // the plan shapes the GPU tests pin, one after the other on one runner (re-pack, upload, free)
  const int rowsLds[][5] = {{64, 1, 1, 16384, 1}, {128, 1, 2, 32768, 3}, {256, 1, 8, 65536, 1}, {512, 1, 4, 49152, 5}, {256, 1, 4, 8192, 40},
                            {256, 4, 4, 65536, 1}, {128, 8, 2, 40960, 2}, {64, 3, 1, 16384, 1}, {512, 2, 8, 32768, 1}};
  for (auto &p : rowsLds)
    if (tbmi_set_plan(runner, p[0], p[1], p[2], p[3], p[4]) == 0) {
      runAll("rows_lds plan");
      for (int mode : {1, 2, 0}) { // tree groups through registers, copied directly, by rule
        EXPECT(tbmi_set_group_staging(runner, mode) == 0, "tbmi_set_group_staging");
        runAll("rows_lds plan, group staging pinned");
      }
    }
  EXPECT(tbmi_set_group_staging(runner, 7) != 0, "tbmi_set_group_staging refuses an unknown mode");
  const int treeParallel[][5] = {{1, 256, 1, 0, 0}, {4, 64, 1, 32768, 7}, {16, 16, 2, 0, 1}, {2, 128, 1, 16384, 0}, {8, 8, 4, 0, 3}, {64, 1, 1, 0, 2}, {1, 1024, 1, 65536, 1}};
  for (auto &p : treeParallel)
    if (tbmi_set_tree_parallel_plan(runner, p[0], p[1], p[2], p[3], p[4]) == 0) runAll("tree_parallel plan");
  const int quantized[][4] = {{8, 4, 0, 1}, {16, 1, 16384, 1}, {4, 2, 32768, 3}, {1, 8, 16384, 1}};
  for (auto &p : quantized)
    if (tbmi_set_quantized_plan(runner, p[0], p[1], p[2], p[3]) == 0) runAll("rank-quantised plan");
  const int rank16[][5] = {{256, 4, 4, 0, 1}, {512, 2, 4, 32768, 1}, {128, 8, 2, 16384, 3}, {64, 1, 1, 16384, 2}};
  for (auto &p : rank16)
    if (tbmi_set_rank16_plan(runner, p[0], p[1], p[2], p[3], p[4]) == 0) runAll("two-byte rank plan");
  if (tbmi_set_global_walk_plan(runner, 256, 4, 3) == 0) runAll("global walk plan");
  double best = 0;
  const long fewInSearch = shimFewRows;
  EXPECT(tbmi_autotune(runner, dx, rows < 96 ? rows : 96, &best) == 0, "tbmi_autotune");
  EXPECT((shimFewRows > fewInSearch) == !!std::strstr(Describe(runner).c_str(), " peelWalks=0 "), "the plan search times the kernel that takes its batch");
  const long fewBefore = shimFewRows;
  EXPECT(tbmi_run_device(runner, dx, dout, 1) == 0 && (shimFewRows > fewBefore || !std::strstr(Describe(runner).c_str(), " peelWalks=0 ")),
         "the plan search ends a pinned plan's hold on small batches");
  runAll("after the plan search");
  MulticlassOutputs(c, runner, dx, rows);
  const std::string file = std::string(std::getenv("TMPDIR") ? std::getenv("TMPDIR") : "/tmp") + "/sanitize_runner.tbamd";
  EXPECT(tbmi_save_compiled_model(runner, file.c_str()) == 0, "tbmi_save_compiled_model");
  const intptr_t again = tbmi_load_compiled_model(file.c_str(), 0);
  EXPECT(again != 0, "tbmi_load_compiled_model");
  if (again) {
    EXPECT(tbmi_run_device(again, dx, dout, rows) == 0, "reloaded runner");
    check("reloaded runner");
    DeleteInferenceRunner(again);
  }
  DeleteInferenceRunner(runner);
  (void)hipFree(dx);
  (void)hipFree(dout);
  (void)hipFree(dids);
}

// A runner made for a small batch, whose plan has many slices: the no-allocation entry point serves the batches that the few-rows
// kernel can take, also above the limit up to which it is the faster form, where the plan's sums do not fit the fixed array.
void NoAllocOfManySums(const Case &c) {
  const intptr_t runner = MakeRunner(c, 512, c.forest.numClasses > 0);
  if (!runner) return;
  const std::string plan = Describe(runner);
  const int64_t limit = std::atoll(plan.c_str() + plan.find("fewRowsLimit=") + std::strlen("fewRowsLimit="));
  const long few = shimFewRows;
  float *dx = nullptr;
  void *out = nullptr;
  const size_t resultBytes = (size_t)c.rows * (size_t)tbmi_result_bytes(runner);
  EXPECT(limit < c.rows, "limit %lld", (long long)limit);
  EXPECT(hipMalloc((void **)&dx, (size_t)c.rows * c.forest.numFeatures * sizeof(float)) == hipSuccess, "hipMalloc");
  EXPECT(hipMalloc(&out, resultBytes) == hipSuccess, "hipMalloc");
  std::memcpy(dx, c.x.data(), (size_t)c.rows * c.forest.numFeatures * sizeof(float));
  EXPECT(tbmi_run_device_noalloc(runner, dx, out, c.rows, nullptr) == 0 && shimFewRows == few + 1, "noalloc of %lld rows, limit %lld",
         (long long)c.rows, (long long)limit);
  std::vector<float> got((size_t)c.rows);
  for (int64_t r = 0; r < c.rows; ++r) got[r] = c.forest.numClasses > 0 ? (float)static_cast<int8_t *>(out)[r] : static_cast<float *>(out)[r];
  Compare(c, got.data(), 0, c.rows, "noalloc of many sums");
  (void)hipFree(dx);
  (void)hipFree(out);
  DeleteInferenceRunner(runner);
}

// Host calls whose n-th launch fails, of one piece and of several: nothing of theirs is under way when they return, and the
// next call is right.
void FailedCalls(const Case &c) {
  const int64_t F = c.forest.numFeatures;
  for (int64_t rows : {std::min<int64_t>(c.rows, 100), std::min<int64_t>(c.rows, 1500), c.rows}) {
    const intptr_t runner = MakeRunner(c, (int32_t)rows, false);
    if (!runner) continue;
    PinOwnPlan(runner);
    std::vector<float> out((size_t)rows);
    void *locked = nullptr;
    EXPECT(hipHostMalloc(&locked, (size_t)rows * F * sizeof(float), 0) == hipSuccess, "hipHostMalloc");
    std::memcpy(locked, c.x.data(), (size_t)rows * F * sizeof(float));
    for (const void *in : {static_cast<const void *>(c.x.data()), static_cast<const void *>(locked)})
      for (long n = 0; n < 6; ++n) {
        shimLaunchesToGo = n;
        const int32_t rc = tbmi_run_host(runner, in, out.data(), rows);
        EXPECT((rc != 0) == (shimLaunchesToGo < 0), "a failed launch is an error");
        shimLaunchesToGo = -1;
        EXPECT(shimBusyStreams(nullptr) == 0, "%lld rows, launch %ld failed: work under way", (long long)rows, n);
        std::fill(out.begin(), out.end(), -1.f);
        EXPECT(tbmi_run_host(runner, in, out.data(), rows) == 0, "the call after a failed one");
        Compare(c, out.data(), 0, rows, "the call after a failed one");
      }
    (void)hipHostFree(locked);
    DeleteInferenceRunner(runner);
  }
}

// All of the case's rows in one device call through every entry point, on the default plan and on plans of several slices
// (which a launch of many blocks splits evenly); calls on the default stream, another stream and the runner's own in turn.
void WholeBatch(const Case &c) {
  const int64_t rows = c.rows, F = c.forest.numFeatures;
  const bool multiclass = c.forest.numClasses > 0;
  const intptr_t runner = MakeRunner(c, (int32_t)rows, multiclass);
  if (!runner) return;
  const std::string plan = Describe(runner);
  const int64_t limit = std::atoll(plan.c_str() + plan.find("fewRowsLimit=") + std::strlen("fewRowsLimit="));
  hipStream_t other = nullptr;
  EXPECT(hipStreamCreateWithFlags(&other, 0) == hipSuccess, "hipStreamCreateWithFlags");
  float *dx = nullptr;
  unsigned char *dout = nullptr;
  const size_t resultBytes = (size_t)rows * (size_t)tbmi_result_bytes(runner);
  EXPECT(hipMalloc((void **)&dx, (size_t)rows * F * sizeof(float)) == hipSuccess, "hipMalloc");
  EXPECT(hipMalloc((void **)&dout, resultBytes) == hipSuccess, "hipMalloc");
  std::memcpy(dx, c.x.data(), (size_t)rows * F * sizeof(float));
  const int plans[][5] = {{0, 0, 0, 0, 0}, {64, 4, 2, 8192, 5}, {64, 16, 4, 16384, 2}, {128, 2, 1, 16384, 3}};
  for (auto &p : plans) {
    if (p[0] && tbmi_set_plan(runner, p[0], p[1], p[2], p[3], p[4]) != 0) continue;
    const auto check = [&](int32_t rc, const char *what) {
      if (rc != 0 && std::strstr(tbmi_last_error(), "scratch memory")) return;
      EXPECT(rc == 0, "%s", what);
      std::vector<float> got((size_t)rows);
      for (int64_t r = 0; r < rows; ++r) got[r] = multiclass ? (float)(int8_t)dout[r] : reinterpret_cast<float *>(dout)[r];
      Compare(c, got.data(), 0, rows, what, other);
      std::memset(dout, 0x5A, resultBytes);
    };
    check(tbmi_run_device_async(runner, dx, dout, rows, nullptr), "async, default stream");
    check(tbmi_run_device_async(runner, dx, dout, rows, other), "async, another stream");
    const long few = shimFewRows, splits = shimSplits, streams = shimStreams;
    check(tbmi_run_device(runner, dx, dout, rows), "run_device");
    const std::string ran = shimFewRows > few ? "few_rows" : shimStreams > streams ? "rank_stream" : shimSplits > splits ? "rows_lds_split" : "";
    const std::string said = Describe(runner).substr(Describe(runner).find("batchKernel=") + std::strlen("batchKernel="));
    EXPECT(ran.empty() ? said.compare(0, 9, "few_rows ") && said.compare(0, 12, "rank_stream ") && said.compare(0, 15, "rows_lds_split ")
                       : said.compare(0, ran.size() + 1, ran + " ") == 0,
           "batchKernel=%s, but the call ran %s", said.c_str(), ran.c_str());
    check(tbmi_run_device_async(runner, dx, dout, rows, nullptr), "async, default stream again");
    check(tbmi_run_device_noalloc(runner, dx, dout, rows, other), "noalloc");
    MulticlassOutputs(c, runner, dx, rows);
  }
  double best = 0, walk = 0, fin = 0, bin = 0;
  (void)tbmi_set_plan(runner, 64, 4, 2, 8192, 1);
  const std::string before = Describe(runner);
  for (int64_t n : {(int64_t)1, rows}) { // a search that fails leaves the plan and its pin (plans no launch of which succeeds are passed over)
    shimNoLaunches = 1;
    const int32_t failed = tbmi_autotune(runner, dx, n, &best);
    shimNoLaunches = 0;
    if (failed) EXPECT(Describe(runner) == before, "after a failed search: %s, before: %s", Describe(runner).c_str(), before.c_str());
    else EXPECT(tbmi_set_plan(runner, 64, 4, 2, 8192, 1) == 0, "tbmi_set_plan");
  }
  EXPECT(tbmi_autotune(runner, dx, std::min<int64_t>(rows, 300), &best) == 0, "tbmi_autotune");
  for (int64_t n : {(int64_t)1, limit, limit + 1, rows}) { // what is timed is what a call runs
    if (n < 1 || n > rows) continue;
    const long few = shimFewRows, streams = shimStreams;
    EXPECT(tbmi_run_device(runner, dx, dout, n) == 0, "run_device");
    const long fewCall = shimFewRows - few, streamCall = shimStreams - streams;
    EXPECT(fewCall == (n <= limit && std::strstr(Describe(runner).c_str(), " peelWalks=0 ")), "%lld rows, limit %lld", (long long)n, (long long)limit);
    EXPECT(tbmi_time_kernels(runner, dx, dout, n, 1, &walk, &fin, &bin) == 0, "tbmi_time_kernels");
    EXPECT(shimFewRows - few == 2 * fewCall && shimStreams - streams == 2 * streamCall, "kernels timed on %lld rows are not the call's", (long long)n);
  }
  EXPECT(tbmi_run_device_async(runner, dx, dout, rows, nullptr) == 0, "async");
  DeleteInferenceRunner(runner);
  (void)hipFree(dx);
  (void)hipFree(dout);
  (void)hipStreamDestroy(other);
}

} // namespace

// Compiled-model files with mutated bytes through tbmi_load_compiled_model and, where one loads, through a host call
// of a few rows: the header's plan, batch size and return type are what a runner is built from.
static int MutatedCompiledModels(const char *path, int iterations) {
  std::ifstream in(path, std::ios::binary);
  const std::vector<char> good((std::istreambuf_iterator<char>(in)), std::istreambuf_iterator<char>());
  EXPECT(!good.empty(), "cannot read %s", path);
  const std::string scratch = std::string(std::getenv("TMPDIR") ? std::getenv("TMPDIR") : "/tmp") + "/mutated.tbamd";
  std::mt19937 rng(13);
  long loaded = 0;
  for (int i = 0; i < iterations; ++i) {
    std::vector<char> bytes = good;
    if (i > 0) {
      const int edits = 1 + (int)(rng() % 3);
      for (int e = 0; e < edits; ++e) {
        const int32_t words[] = {0, 1, -1, 2, 3, 7, 8, 9, 63, 64, 65, 255, 1000, 1024, 65536, 1 << 20, 1 << 30, INT32_MIN};
        const int32_t w = words[rng() % 18];
        const size_t limit = rng() % 4 ? std::min<size_t>(bytes.size(), 140) : bytes.size(); // mostly the header
        const size_t p = (rng() % limit) & ~(size_t)3;
        std::memcpy(bytes.data() + p, &w, std::min<size_t>(4, bytes.size() - p));
      }
    }
    {
      std::ofstream out(scratch, std::ios::binary | std::ios::trunc);
      out.write(bytes.data(), (std::streamsize)bytes.size());
    }
    const intptr_t runner = tbmi_load_compiled_model(scratch.c_str(), 0);
    if (!runner) {
      EXPECT(i > 0, "the intact compiled model was refused: %s", tbmi_last_error());
      continue;
    }
    ++loaded;
    const int32_t F = GetRowSize(runner);
    EXPECT(F > 0 && F < (1 << 20), "row size %d of a loaded model", F);
    const int64_t rows = 70;
    std::vector<float> x((size_t)rows * F, 0.25f);
    std::vector<unsigned char> out((size_t)rows * (size_t)tbmi_result_bytes(runner), 0xEE); // exactly what the call may write
    (void)tbmi_run_host(runner, x.data(), out.data(), rows); // may be refused; must not overrun
    DeleteInferenceRunner(runner);
  }
  std::printf("mutated compiled models: %ld of %d loaded\n", loaded, iterations);
  return gFailures;
}

// A classifier whose tree threads' own classes leave their meeting place to the groups: shapes in which they meet again, pinned with
// the group size kept, find that place free - straight away, from a compiled-model file, and with the fields of older files, whose one
// group size is either that without the place or that with it.
void KeptGroupSize(const Case &c) {
  const auto field = [](const std::string &text, const char *name) {
    const size_t at = text.find(std::string(" ") + name + "=");
    return at == std::string::npos ? -1 : std::atoi(text.c_str() + at + std::strlen(name) + 2);
  };
  const std::string file = std::string(std::getenv("TMPDIR") ? std::getenv("TMPDIR") : "/tmp") + "/kept_group_size.tbamd";
  std::vector<float> out((size_t)c.rows);
  int meet = 0, own = 0;
  for (int from = 0; from < 4; ++from) {
    intptr_t runner = MakeRunner(c, 40731, false);
    const std::string chosen = Describe(runner);
    const int threads = field(chosen, "treeThreads"), group = field(chosen, "groupBytes");
    if (from > 0) {
      EXPECT(tbmi_save_compiled_model(runner, file.c_str()) == 0, "tbmi_save_compiled_model");
      DeleteInferenceRunner(runner);
      if (from > 1) { // version 5: 14 words of plan behind 48 bytes
        std::ifstream in(file, std::ios::binary);
        std::string bytes((std::istreambuf_iterator<char>(in)), std::istreambuf_iterator<char>());
        in.close();
        bytes[8] = 5;
        if (from == 3) bytes.replace(48 + 5 * 4, 4, bytes, 48 + 14 * 4, 4);
        bytes.erase(48 + 14 * 4, 4);
        std::ofstream(file, std::ios::binary) << bytes;
      }
      runner = tbmi_load_compiled_model(file.c_str(), 0);
      EXPECT(runner != 0, "tbmi_load_compiled_model");
      const std::string loaded = Describe(runner);
      EXPECT((loaded == chosen) == (from != 2) && field(loaded, "groupBytes") <= group, "%s\n%s", chosen.c_str(), loaded.c_str());
    }
    for (int k : {1, 2, 4, 8})
      for (int slices : {1, 4}) {
        EXPECT(tbmi_set_plan(runner, 0, threads, k, 0, slices) == 0, "interleave %d, %d slices", k, slices);
        const std::string plan = Describe(runner);
        ++(field(plan, "ownClasses") ? own : meet);
        EXPECT(field(plan, "interleave") == k && field(plan, "ldsBytes") <= 160 * 1024, "%s", plan.c_str());
        EXPECT(tbmi_run_host(runner, c.x.data(), out.data(), c.rows) == 0, "tbmi_run_host");
        Compare(c, out.data(), 0, c.rows, "a plan of another interleave");
      }
    // a size that the caller names is kept whoever the classes are
    EXPECT(tbmi_set_plan(runner, 0, threads, 2, 16384, 1) == 0 && field(Describe(runner), "groupBytes") == 16384, "%s", Describe(runner).c_str());
    DeleteInferenceRunner(runner);
  }
  EXPECT(meet > 0 && own > 0, "%d plans with classes that meet, %d without", meet, own);
}

int main(int argc, char **argv) {
  // argv: pairs of <model.json> <rows>, or --mutate <compiled model> <iterations>
  if (argc == 4 && std::strcmp(argv[1], "--mutate") == 0) {
    if (int rc = MutatedCompiledModels(argv[2], std::atoi(argv[3]))) return rc;
    std::printf("few-rows launches %ld\n", shimFewRows);
    std::printf("ok\n");
    return 0;
  }
  std::mt19937 rng(7);
  std::normal_distribution<float> normal(0.f, 1.f);
  for (int a = 1; a + 1 < argc; a += 2) {
    Case c;
    c.path = argv[a];
    c.rows = std::atoll(argv[a + 1]);
    c.forest = LoadForest(argv[a]);
    const int64_t F = c.forest.numFeatures;
    c.x.resize((size_t)c.rows * F);
    for (auto &v : c.x) v = normal(rng);
    c.expected.resize((size_t)c.rows);
    for (int64_t r = 0; r < c.rows; ++r) c.expected[r] = Predict(c.forest, c.x.data() + r * F, nullptr);
    if (std::getenv("SANITIZE_NOALLOC")) {
      NoAllocOfManySums(c);
      continue;
    }
    if (std::getenv("SANITIZE_SHAPES")) {
      KeptGroupSize(c);
      continue;
    }
    HostEntryPoints(c);
    HostEntryPoints(c, true);
    WholeBatch(c);
    FailedCalls(c);
    DeviceEntryPoints(c, std::min<int64_t>(c.rows, 203));
    if (!Quick()) {
      const std::string profile =
          WriteProfile(c, std::string(std::getenv("TMPDIR") ? std::getenv("TMPDIR") : "/tmp") + "/sanitize_profile.csv");
      // (every tile layout on every model; the profiled variants of the odd sizes on the first model only)
      for (int32_t tileSize : {2, 3, 4, 5, 8}) {
        DeviceEntryPoints(c, std::min<int64_t>(c.rows, 203), tileSize);
        if (a > 1 && (tileSize == 3 || tileSize == 5)) continue;
        DeviceEntryPoints(c, std::min<int64_t>(c.rows, 203), tileSize, 1, profile.c_str(), true);
        if (a > 1 && tileSize != 4) continue;
        DeviceEntryPoints(c, std::min<int64_t>(c.rows, 203), tileSize, 2, profile.c_str(), false);
      }
      DeviceEntryPoints(c, std::min<int64_t>(c.rows, 203), 1, 1, profile.c_str(), true); // scalar nodes, peeled walks
      const intptr_t options = CreateCompilerOptions();
      Set_batchSize(options, 64);
      Set_tileSize(options, 9);
      EXPECT(CreateInferenceRunner(c.path.c_str(), "", options) == 0 && std::strstr(tbmi_last_error(), "tile size 9"),
             "tile size 9 must be refused");
      DeleteCompilerOptions(options);
    }
    std::printf("%s: %lld rows done, %d failures so far\n", argv[a], (long long)c.rows, gFailures);
    std::fflush(stdout);
  }
  // error paths keep their hands off the caller's buffers
  EXPECT(tbmi_run_device(0, nullptr, nullptr, 4) == -1, "null runner");
  EXPECT(CreateInferenceRunner("/nonexistent/model.json", "", 0) == 0, "missing options");
  if (gFailures) return 1;
  std::printf("launches: few-rows %ld, split %ld, stream %ld, deferred %ld\nok\n", shimFewRows, shimSplits, shimStreams, shimDeferred);
  return 0;
}
