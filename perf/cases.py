"""What users of this library have it do: batch inference of tree ensembles, from one row to a million.

A case names a forest (trees, depth, how bushy, features, classes), a batch and the entry point the rows go
through.  The forests are those of the five benchmark configurations (treebeard_amd/synth.py) and of the tests,
grown here level by level with numpy: seeded by the case's own numbers, because a program keeps its model while
its rows change.  `prepare` makes rows from the seed alone and hands out the runner a program would have open;
`run` is one call on them.

Entry points ("call"):
  stream   rows in device memory, kernels enqueued on torch's current stream (run_device_async)
  scores   rows in device memory, a classifier's class ids, per-class sums and softmax (run_device_multiclass)
  host     numpy in, numpy out, one compiled batch per call (RunInference)
  batches  numpy in, numpy out, several compiled batches per call (RunInferenceOnMultipleBatches)
"""
import collections
import json
import math
import os
import tempfile

import numpy as np
import torch

from treebeard_amd import treebeard

# The largest listed work, in (row, tree, level) steps and in feature values; draws stay below both.
MOST_STEPS = (1 << 20) * 8000
MOST_VALUES = (1 << 18) * 2000


def _case(name, call, rows, trees, depth, features, left=0.8, right=0.8, levels=4096, classes=0, sigmoid=False, hot=False,
          tile=1, batch=0):
    """left / right: chance that a left / right child splits again; levels: distinct split values per feature (0:
    any); hot: most rows follow the left spine; tile: CompilerOptions' tile size; batch: compiled batch (0: rows)."""
    case = {"call": call, "rows": rows, "trees": trees, "depth": depth, "features": features, "left": left, "right": right,
            "levels": levels, "classes": classes, "sigmoid": sigmoid, "hot": hot, "tile": tile, "batch": batch or rows}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one request of an online service: a row that is already on the device, a binary classifier of the headline size
        _case("one_row", "stream", 1, 1000, 8, 28, sigmoid=True),
        # a script that scores small numpy batches with the reference's RunInference (its own benchmark starts at 512 rows)
        _case("host_512", "host", 512, 100, 6, 8, left=1.0, right=1.0),
        # a micro-batching server: thousands of rows per launch, too few to fill the chip with one lane per row
        _case("batch_4096", "stream", 4096, 1000, 8, 28, sigmoid=True),
        # a ragged mid-size batch of a regressor with a hundred deep-ish trees on 90 features
        _case("ragged_50001", "stream", 50001, 100, 9, 90),
        # the headline: bulk scoring of 2^20 rows in device memory
        _case("bulk_1m", "stream", 1 << 20, 1000, 8, 28, sigmoid=True),
        # bulk class ids of an eight-class model with complete trees, a few continuous features and many 0/1 ones
        _case("classes_1m", "stream", 1 << 20, 800, 6, 54, left=1.0, right=1.0, classes=8),
        # class ids with sums and probabilities, odd number of rows
        _case("scores_65537", "scores", 65537, 800, 6, 54, left=1.0, right=1.0, classes=8),
        # wide rows: 2000 features, where reading the rows is what memory has to do
        _case("wide_256k", "stream", 1 << 18, 1000, 8, 2000, left=0.85, right=0.85, levels=0),
        # skewed trees and rows: long left spines that most rows follow
        _case("skewed_1m", "stream", 1 << 20, 800, 12, 90, left=0.9, right=0.3, hot=True),
        # callers that keep the reference's habitual tile size 8
        _case("tile8_64k", "stream", 1 << 16, 1000, 8, 28, sigmoid=True, tile=8),
        # a forest of few, deep trees, each too big for a tree group in local memory
        _case("deep_64k", "stream", 1 << 16, 40, 16, 28, left=0.88, right=0.88, levels=0),
        # bulk scoring from numpy: 16 compiled batches in one call, the rows cross the host link
        _case("host_batches", "batches", 1 << 18, 1000, 8, 28, sigmoid=True, batch=1 << 14),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("small", "host", "plain", "plain", "plain", "classes", "scores", "wide", "skewed", "tiled", "deep", "batches"))
    trees, depth, features = _log_int(rng, 50, 1000), rng.randint(4, 9), _log_int(rng, 5, 150)
    split = round(rng.uniform(0.75, 1.0), 3) if depth <= 8 else 0.8
    levels, sigmoid = rng.choice((0, 255, 4096)), rng.random() < 0.5
    rows, more, call = _log_int(rng, 4000, 1 << 20), {}, "stream"
    if kind == "small":
        rows = _log_int(rng, 1, 4096)
    elif kind == "host":
        call, rows = "host", _log_int(rng, 1, 16384)
    elif kind in ("classes", "scores"):
        call, sigmoid, more = ("scores" if kind == "scores" else "stream"), False, {"classes": rng.randint(3, 12)}
    elif kind == "wide":
        features, rows, levels = _log_int(rng, 600, 2000), _log_int(rng, 4000, 1 << 18), rng.choice((0, 255))
    elif kind == "skewed":
        depth, more = rng.randint(9, 12), {"hot": True}
    elif kind == "tiled":
        rows, more = _log_int(rng, 1000, 1 << 17), {"tile": rng.randint(2, 8)}
    elif kind == "deep":
        rows, trees, depth, split, levels = _log_int(rng, 1000, 1 << 16), rng.randint(10, 40), rng.randint(15, 16), 0.88, 0
    elif kind == "batches":
        batch = 1 << rng.randint(9, 14)
        call, rows, more = "batches", batch * max(1, min(rows, 1 << 18) // batch), {"batch": batch}
    if call != "batches":
        rows = max(1, min(rows, MOST_STEPS // (trees * depth), MOST_VALUES // features))
    left, right = (0.9, 0.3) if kind == "skewed" else (split, split)
    return _case(None, call, rows, trees, depth, features, left=left, right=right, levels=levels, sigmoid=sigmoid, **more)


# ---- the model -------------------------------------------------------------------------------------------

def _grow(rng, case):
    """Level-order forests, all trees at once: (owner tree, id in the tree, left child or -1) of every node, by (owner, id)."""
    trees, depth = case["trees"], case["depth"]
    owner, ident = np.arange(trees), np.zeros(trees, np.int64)
    chance = np.ones(trees)
    used = np.ones(trees, np.int64)                         # ids handed out per tree
    levels = []
    for level in range(depth + 1):
        splits = (rng.random(owner.size) < chance) if level < depth else np.zeros(owner.size, bool)
        parents = owner[splits]
        first = np.searchsorted(parents, np.arange(trees))  # parents are sorted by tree
        left = np.full(owner.size, -1, np.int64)
        left[splits] = used[parents] + 2 * (np.arange(parents.size) - first[parents])
        levels.append((owner, ident, left))
        used = used + 2 * np.bincount(parents, minlength=trees)
        ident = np.repeat(left[splits], 2)
        ident[1::2] += 1
        owner = np.repeat(parents, 2)
        chance = np.tile([case["left"], case["right"]], parents.size)
    owner, ident, left = (np.concatenate(part) for part in zip(*levels))
    order = np.lexsort((ident, owner))
    return owner[order], left[order]


def _binary_features(case):
    """Of a classifier's features all but ten are 0/1 indicators (as in its benchmark configuration)."""
    return max(0, case["features"] - 10) if case["classes"] else 0


def _write_model(case, path):
    rng = np.random.Generator(np.random.PCG64([7, case["trees"], case["depth"], case["features"], case["levels"]]))
    owner, left = _grow(rng, case)
    inner = left >= 0
    feature = np.where(inner, rng.integers(0, case["features"], left.size), 0)
    threshold = rng.standard_normal(left.size).astype(np.float32)
    if case["levels"]:                                      # split values on a grid of quantiles, as histogram training leaves them
        grid = np.sort(rng.standard_normal((case["levels"], case["features"])).astype(np.float32), axis=0)
        threshold = grid[rng.integers(0, case["levels"], left.size), feature]
    threshold[feature >= case["features"] - _binary_features(case)] = 0.5
    value = np.where(inner, threshold, rng.normal(0.0, 0.05, left.size).astype(np.float32))
    ends = np.flatnonzero(np.diff(owner, append=case["trees"])) + 1
    trees, begin = [], 0
    for end in ends:
        here = slice(begin, end)
        begin = end
        trees.append({"left_children": left[here].tolist(), "right_children": np.where(inner[here], left[here] + 1, -1).tolist(),
                      "split_conditions": value[here].tolist(), "split_indices": feature[here].tolist(),
                      "tree_param": {"num_nodes": str(end - here.start), "num_feature": str(case["features"])}})
    objective = "multi:softmax" if case["classes"] else "binary:logistic" if case["sigmoid"] else "reg:squarederror"
    info = [t % case["classes"] if case["classes"] else 0 for t in range(case["trees"])]
    with open(path, "w") as out:
        out.write(json.dumps({"learner": {
            "feature_types": ["float"] * case["features"], "objective": {"name": objective},
            "learner_model_param": {"base_score": "5E-1", "num_class": str(case["classes"]), "num_feature": str(case["features"])},
            "gradient_booster": {"model": {"gbtree_model_param": {"num_trees": str(case["trees"])}, "tree_info": info,
                                           "trees": trees}}}}))


_runners = collections.OrderedDict()


def _runner(case):
    """The runner a program keeps open for its model and batch; the last two stay open here."""
    key = json.dumps({k: v for k, v in case.items() if k not in ("name", "rows", "hot")}, sort_keys=True)
    if key not in _runners:
        options = treebeard.CompilerOptions(case["batch"], case["tile"])
        if case["classes"]:                                 # class ids as bytes
            options.SetReturnTypeWidth(8)
            options.SetReturnTypeIsFloatType(False)
        with tempfile.TemporaryDirectory() as folder:
            path = os.path.join(folder, "model.json")
            _write_model(case, path)
            _runners[key] = treebeard.TreebeardInferenceRunner.FromModelFile(path, "", options)
        while len(_runners) > 2:
            _runners.popitem(last=False)
    _runners.move_to_end(key)
    return _runners[key]


# ---- one case --------------------------------------------------------------------------------------------

def prepare(case, seed):
    rows, features = case["rows"], case["features"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(rows, features, generator=gen, device="cuda")
    binary = _binary_features(case)
    if binary:
        x[:, features - binary:] = (torch.rand(rows, binary, generator=gen, device="cuda") < 0.1).float()
    if case["hot"]:                                         # about 80 % of the rows from a low population
        low = torch.rand(rows, 1, generator=gen, device="cuda") < 0.8
        x = torch.where(low, x * 0.5 - 2.0, x)
    state = {"call": case["call"], "rows": rows, "runner": _runner(case)}
    if case["call"] in ("host", "batches"):
        state["x"] = x.cpu().numpy()
        return state
    state["x"] = x
    state["out"] = torch.zeros(rows, dtype=torch.int8 if case["classes"] else torch.float32, device="cuda")
    if case["call"] == "scores":
        state["sums"] = torch.zeros(rows, case["classes"], device="cuda")
        state["probabilities"] = torch.zeros(rows, case["classes"], device="cuda")
    torch.cuda.synchronize()                                # (run_device_multiclass runs on the runner's own stream)
    return state


def run(state):
    runner, x = state["runner"], state["x"]
    if state["call"] == "host":
        return runner.RunInference(x, runner.result_dtype())
    if state["call"] == "batches":
        return runner.RunInferenceOnMultipleBatches(x, runner.result_dtype())
    if state["call"] == "scores":
        runner.run_device_multiclass(x.data_ptr(), state["rows"], state["out"].data_ptr(), state["sums"].data_ptr(),
                                     state["probabilities"].data_ptr())
        return state["out"], state["sums"], state["probabilities"]
    runner.run_device_async(x.data_ptr(), state["out"].data_ptr(), state["rows"], torch.cuda.current_stream().cuda_stream)
    return state["out"]


def _visits(case):
    """Internal nodes a row visits on average over the forest, if every split sends half of the rows either way."""
    split = 0.5 * (case["left"] + case["right"])
    return case["trees"] * sum(split ** level for level in range(case["depth"]))


def work(case):
    """Rows in, results out, the model (8 bytes a node) once; a comparison per visited node and an addition per tree."""
    rows = case["rows"]
    nodes = case["trees"] * (1 + 2 * sum((case["left"] + case["right"]) ** level for level in range(case["depth"])))
    result = 1 + 8 * case["classes"] if case["call"] == "scores" else 1 if case["classes"] else 4
    return {"bytes": rows * (4 * case["features"] + result) + 8 * nodes, "flops": rows * (_visits(case) + case["trees"])}


def tolerance(case):
    """Leaf values are added in 64 bits and rounded once to 32.  A class id may differ where two classes' rounded sums
    tie, which another order of the additions can decide the other way for a row or two of a million."""
    limits = {"rel": 1e-6, "max": 1e-5}
    if case["classes"]:
        limits["differ"] = 3e-6
    return limits
