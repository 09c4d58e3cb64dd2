"""Forests whose trees do not fit LDS whole, walked with deferred tails: leaf for leaf the global-memory walk's predictions, over
the three block shapes, odd batches, rows of infinities and NaN, the four comparisons."""
import json

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle, model_io  # noqa: E402
from treebeard_amd import synth  # noqa: E402

from onnx_writer import write_onnx  # noqa: E402
from test_gpu_parity import RTOL_SUM, gpu_predict, make_runner  # noqa: E402
from test_gpu_plan_shapes import full_tree  # noqa: E402


def deep_model(path, features, trees=9, leaf=lambda rng: rng.normal(0.0, 0.1), depth=13, **kind):
    rng = np.random.Generator(np.random.PCG64(features))
    split = lambda: (rng.integers(0, features), rng.normal())
    grown = [synth._grow_tree(rng, depth, lambda d, s: 1.0, split, lambda: leaf(rng))]
    grown += [synth._grow_tree(rng, int(rng.integers(0, 15)), lambda d, s: 0.9, split, lambda: leaf(rng), force_root=False)
              for _ in range(trees - 1)]
    synth.write_xgboost_json(path, grown, features, **kind)
    return path


def batch_of(runner, more=0):
    """The first batch above the few-rows limit, and `more`."""
    return int(runner.describe_plan().split("fewRowsLimit=")[1].split()[0]) + 1 + more


# 51 / 52, 102 / 104: the last features of a shape, the first of the next; 254: the widest row tile
@pytest.mark.parametrize("features", [1, 12, 51, 52, 102, 104, 254])
def test_deep_walk_matches_the_oracle(tmp_path, features):
    path = deep_model(tmp_path / "deep.json", features)
    forest = model_io.load_xgboost_json(path)
    small = make_runner(path, 100)
    for more in (0, 30000):
        rows = batch_of(small, more)
        runner = make_runner(path, rows)
        assert "batchKernel=deep_walk" in runner.describe_plan()
        x = np.random.Generator(np.random.PCG64(rows)).normal(size=(rows, features)).astype(np.float32)
        x[0, ::2] = np.inf
        x[1, :] = -np.inf
        x[2, ::3] = np.nan
        got = gpu_predict(runner, x)
        np.testing.assert_allclose(got, cpu_oracle.predict(forest, x)[0], rtol=RTOL_SUM, atol=1e-7)
        out = torch.zeros(rows, device="cuda")
        dx = torch.from_numpy(x).cuda()
        stream = torch.cuda.current_stream()
        for call in (runner.run_device_async, runner.run_device_noalloc):
            out.zero_()
            call(dx.data_ptr(), out.data_ptr(), rows, stream.cuda_stream)
            stream.synchronize()
            np.testing.assert_array_equal(out.cpu().numpy(), got)
        runner.set_global_walk_plan(256, 4, 1)
        assert "batchKernel=global_walk" in runner.describe_plan()
        np.testing.assert_allclose(gpu_predict(runner, x), got, rtol=1e-6, atol=1e-7)


@pytest.mark.parametrize("mode", ["BRANCH_LT", "BRANCH_LEQ", "BRANCH_GT", "BRANCH_GEQ"])
def test_comparison_modes(tmp_path, mode):
    rng = np.random.Generator(np.random.PCG64(4))
    trees = []
    for depth, p in ((13, 1.0), (14, 0.85), (5, 1.0)):
        t = synth._grow_tree(rng, depth, lambda d, s: p, lambda: (rng.integers(0, 12), np.round(rng.normal(), 1)), rng.normal)
        trees.append((t.value, t.feature, t.left, t.right))
    path = str(tmp_path / "deep.onnx")
    write_onnx(path, trees, mode=mode)
    rows = batch_of(make_runner(path, 100, "onnx_file", 12), 3000)
    runner = make_runner(path, rows, "onnx_file", 12)
    assert "batchKernel=deep_walk " in runner.describe_plan()
    x = np.round(rng.normal(size=(rows, 12)), 1).astype(np.float32)  # (values on the thresholds)
    np.testing.assert_allclose(gpu_predict(runner, x), cpu_oracle.predict(model_io.load_onnx(path, 12), x)[0], rtol=RTOL_SUM, atol=1e-6)


def test_plan_search_of_a_deep_forest(tmp_path):
    path = deep_model(tmp_path / "deep.json", 20, objective="binary:logistic")
    forest = model_io.load_xgboost_json(path)
    rows = batch_of(make_runner(path, 100), 5000)
    runner = make_runner(path, rows)
    x = np.random.Generator(np.random.PCG64(3)).normal(size=(rows, 20)).astype(np.float32)
    dx = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    runner.autotune(dx.data_ptr(), rows)
    assert "batchKernel=deep_walk" in runner.describe_plan()
    np.testing.assert_allclose(gpu_predict(runner, x), cpu_oracle.predict(forest, x)[0], rtol=0, atol=1e-6)


def test_nodes_that_no_walk_reaches(tmp_path):
    """Leaves behind those of the trees, as pruning leaves them, in trees that are cut and in trees that stay whole."""
    rng = np.random.Generator(np.random.PCG64(11))
    trees = [full_tree(rng, nodes, 12) for nodes in (16383, 9001, 31, 1, 301)]
    for tree, more in zip(trees, (2, 700, 9000, 1, 1)):
        tree.left += [-1] * more
        tree.right += [-1] * more
        tree.parent += [0] * more
        tree.feature += [0] * more
        tree.value += [100.0] * more
    path = str(tmp_path / "pruned.json")
    synth.write_xgboost_json(path, trees, 12)
    rows = batch_of(make_runner(path, 100), 2000)
    runner = make_runner(path, rows)
    assert "batchKernel=deep_walk " in runner.describe_plan()
    x = rng.standard_normal((rows, 12), dtype=np.float32)
    np.testing.assert_allclose(gpu_predict(runner, x), cpu_oracle.predict(model_io.load_xgboost_json(path), x)[0], rtol=RTOL_SUM, atol=1e-7)


# 260 trees of 16128 tail nodes each are the most the tail array holds; 263 were the fewest that an estimate let through
@pytest.mark.parametrize("trees,kernel", [(260, "deep_walk"), (263, "global_walk")])
def test_as_many_tail_nodes_as_there_are_places(tmp_path, trees, kernel):
    """The same tree over and over: the sum is so many times one tree's leaf."""
    rng = np.random.Generator(np.random.PCG64(12))
    one, many = str(tmp_path / "one.json"), str(tmp_path / "many.json")
    synth.write_xgboost_json(one, [full_tree(rng, 16383, 28)], 28)
    doc = json.load(open(one))
    model = doc["learner"]["gradient_booster"]["model"]
    tree = json.dumps({k: v for k, v in model["trees"][0].items()
                       if k in ("left_children", "right_children", "split_conditions", "split_indices", "tree_param")})
    model["gbtree_model_param"]["num_trees"], model["tree_info"], model["trees"] = str(trees), [0] * trees, ["TREES"]
    with open(many, "w") as out:
        out.write(json.dumps(doc).replace('"TREES"', ",".join([tree] * trees)))
    runner = make_runner(many, 5000)
    assert "batchKernel=%s " % kernel in runner.describe_plan(), runner.describe_plan()
    x = rng.standard_normal((5000, 28), dtype=np.float32)
    leaf = cpu_oracle.predict(model_io.load_xgboost_json(one), x)[0].astype(np.float64) - 0.5
    # (one tree's prediction is rounded to 32 bits next to 0.5, half a unit in the last place 3e-8, and taken `trees` times)
    np.testing.assert_allclose(gpu_predict(runner, x), 0.5 + trees * leaf, rtol=RTOL_SUM, atol=trees * 6e-8)


def test_plan_description_has_the_shape_of_the_deep_walk(tmp_path):
    runner = make_runner(deep_model(tmp_path / "deep.json", 20), 60000)
    fields = dict(item.split("=", 1) for item in runner.describe_plan().split() if "=" in item)
    assert fields["batchKernel"] == "deep_walk" and fields["kernel"] == "global_walk"
    assert fields["deepRowsPerBlock"] == "256" and fields["deepTreeThreads"] == "4" and fields["deepInterleave"] == "2"
    assert int(fields["deepTreesDeferred"]) > 0 and int(fields["deepTreeSlices"]) in (1, 2)
    assert 0 < int(fields["deepLockStepSteps"]) < 9 * 14 and 0 < int(fields["deepLdsBytes"]) <= 80 * 1024
    runner.set_global_walk_plan(256, 4, 1)
    assert "deepRowsPerBlock" not in runner.describe_plan()
