"""Batches of a few rows (one launch, a lane per row and tree) against the oracle: the edges of its range and of its
blocks, every entry point, classifiers with all their outputs, non-finite rows, trees that are single leaves."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle, model_io  # noqa: E402
from treebeard_amd import synth  # noqa: E402

from test_gpu_parity import ATOL_PROB, RTOL_SUM, gpu_predict, make_runner  # noqa: E402


def limit_of(runner):
    return int(runner.describe_plan().split("fewRowsLimit=")[1].split()[0])


def close(forest, got, expected):
    if forest.num_classes > 0:
        np.testing.assert_array_equal(got.astype(np.float32), expected)
    elif forest.transform == model_io.SIGMOID:
        np.testing.assert_allclose(got, expected, rtol=0, atol=ATOL_PROB)
    else:
        np.testing.assert_allclose(got, expected, rtol=RTOL_SUM, atol=0)


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5])
def test_few_rows_match_the_oracle(synth_model, k):
    forest = model_io.load_xgboost_json(synth_model(k))
    runner = make_runner(synth_model(k), 64)
    limit = limit_of(runner)
    assert limit >= 64
    sizes = sorted({1, 2, 63, 64, 255, 256, 257, limit - 1, limit, limit + 1})
    x = synth.CONFIGS[k].batch_rows(limit + 1, seed_offset=5)
    x[0, ::2] = np.inf
    x[1, :] = -np.inf
    x[2, ::3] = np.nan
    expected = cpu_oracle.predict(forest, x)[0]
    for rows in [s for s in sizes if 0 < s <= limit + 1]:
        close(forest, gpu_predict(runner, x[:rows]), expected[:rows])
    stream = torch.cuda.current_stream()
    out = torch.zeros(limit, dtype=torch.int8 if forest.num_classes else torch.float32, device="cuda")
    dx = torch.from_numpy(x).cuda()
    for call in (runner.run_device_async, runner.run_device_noalloc):
        out.zero_()
        call(dx.data_ptr(), out.data_ptr(), limit, stream.cuda_stream)
        stream.synchronize()
        close(forest, out.cpu().numpy(), expected[:limit])
    close(forest, runner.RunInference(x[:64], runner.result_dtype()), expected[:64])
    close(forest, runner.run_host(x[:limit]), expected[:limit])


def test_few_rows_of_a_classifier_with_sums_and_probabilities(synth_model):
    forest = model_io.load_xgboost_json(synth_model(3))
    runner = make_runner(synth_model(3), 300)
    rows, classes = 300, forest.num_classes
    assert rows <= limit_of(runner)
    x = synth.CONFIGS[3].batch_rows(rows, seed_offset=6)
    pred, sums = cpu_oracle.predict(forest, x)
    dx = torch.from_numpy(x).cuda()
    ids = torch.full((rows,), -1, dtype=torch.int8, device="cuda")
    margins, probabilities = (torch.full((rows, classes), -1.0, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    runner.run_device_multiclass(dx.data_ptr(), rows, ids.data_ptr(), margins.data_ptr(), probabilities.data_ptr())
    np.testing.assert_array_equal(ids.cpu().numpy().astype(np.float32), pred)
    np.testing.assert_allclose(margins.cpu().numpy(), sums, rtol=RTOL_SUM, atol=1e-7)
    z = np.exp(sums.astype(np.float64) - sums.max(axis=1, keepdims=True))
    np.testing.assert_allclose(probabilities.cpu().numpy(), z / z.sum(axis=1, keepdims=True), rtol=0, atol=ATOL_PROB)


def test_few_rows_of_small_and_lopsided_trees(tmp_path):
    """Single leaves, one split, a spine of 20 levels: every slot of a block and every exit is some tree's leaf."""
    rng = np.random.Generator(np.random.PCG64(3))

    def draw_split():
        return rng.integers(0, 5), rng.standard_normal()

    def draw_leaf():
        return rng.normal()
    trees = [synth._grow_tree(rng, depth, lambda d, s: 0.6, draw_split, draw_leaf, force_root=depth > 0) for depth in (0, 1, 2, 3, 4, 5, 6, 7) for _ in range(9)]
    trees += [synth._grow_tree(rng, 20, lambda d, s: 1.0 if s == side else 0.1, draw_split, draw_leaf) for side in (0, 1)]
    for count in (1, len(trees)):
        path = str(tmp_path / ("model%d.json" % count))
        synth.write_xgboost_json(path, trees[:count], 5)
        forest = model_io.load_xgboost_json(path)
        x = rng.standard_normal((301, 5), dtype=np.float32)
        expected = cpu_oracle.predict(forest, x)[0]
        runner = make_runner(path, 301)
        assert limit_of(runner) >= 301
        for rows in (1, 5, 301):
            close(forest, gpu_predict(runner, x[:rows]), expected[:rows])


def test_calls_on_the_default_and_other_streams_follow_each_other(synth_model):
    """A call on the default stream leaves its event to the next call on another stream."""
    forest = model_io.load_xgboost_json(synth_model(2))
    runner = make_runner(synth_model(2), 5000)
    x = synth.CONFIGS[2].batch_rows(5000, seed_offset=2)
    expected = cpu_oracle.predict(forest, x)[0]
    dx = torch.from_numpy(x).cuda()
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    for rows in (5000, 100):
        outs = [torch.zeros(rows, device="cuda") for _ in range(4)]
        torch.cuda.synchronize()
        for i, out in enumerate(outs):
            runner.run_device_async(dx.data_ptr(), out.data_ptr(), rows, None if i % 2 == 0 else other.cuda_stream)
        torch.cuda.synchronize()
        for out in outs:
            np.testing.assert_allclose(out.cpu().numpy(), expected[:rows], rtol=0, atol=ATOL_PROB)
        runner.run_device_async(dx.data_ptr(), outs[0].data_ptr(), rows, None)
        runner.run_device(dx.data_ptr(), outs[1].data_ptr(), rows)
        np.testing.assert_allclose(outs[1].cpu().numpy(), expected[:rows], rtol=0, atol=ATOL_PROB)


@pytest.mark.parametrize("classes,trees,features,depth", [(2, 2, 4, 3), (3, 3, 2, 6)])
def test_small_classifiers_at_their_limit_and_far_beyond(tmp_path, classes, trees, features, depth):
    """Few trees: a block has few waves for its rows.  Every row's four outputs are written, on both sides of the limit."""
    rng = np.random.Generator(np.random.PCG64(classes))

    def draw_split():
        return rng.integers(0, features), rng.standard_normal()
    path = str(tmp_path / "small.json")
    synth.write_xgboost_json(path, [synth._grow_tree(rng, depth, lambda d, s: 1.0, draw_split, lambda: rng.normal()) for _ in range(trees)],
                             features, objective="multi:softmax", num_class=classes, tree_info=[t % classes for t in range(trees)])
    forest = model_io.load_xgboost_json(path)
    runner = make_runner(path, 1024)
    limit = limit_of(runner)
    x = rng.standard_normal((393216, features), dtype=np.float32)
    pred, sums = cpu_oracle.predict(forest, x, threads=8)
    z = np.exp(sums.astype(np.float64) - sums.max(axis=1, keepdims=True))
    dx = torch.from_numpy(x).cuda()
    for rows in sorted({limit, limit + 1, 262144, 262145, 393216}):
        ids = torch.full((rows,), -1, dtype=torch.int8, device="cuda")
        margins, probabilities = (torch.full((rows, classes), -1.0, device="cuda") for _ in range(2))
        torch.cuda.synchronize()
        runner.run_device_multiclass(dx.data_ptr(), rows, ids.data_ptr(), margins.data_ptr(), probabilities.data_ptr())
        np.testing.assert_array_equal(ids.cpu().numpy().astype(np.float32), pred[:rows])
        np.testing.assert_allclose(margins.cpu().numpy(), sums[:rows], rtol=RTOL_SUM, atol=1e-7)
        np.testing.assert_allclose(probabilities.cpu().numpy(), (z / z.sum(axis=1, keepdims=True))[:rows], rtol=0, atol=ATOL_PROB)
        close(forest, gpu_predict(runner, x[:rows]), pred[:rows])
