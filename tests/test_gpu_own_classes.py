"""Classifiers whose classes are each one tree thread's: numbers of classes below, around and above the tree threads', classes without trees or with
more than others, equal sums (the larger class id), every output, slices, even splits, groups of one and several rounds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle, model_io  # noqa: E402
from treebeard_amd import synth  # noqa: E402

from test_gpu_parity import RTOL_SUM, gpu_leaf_ids, gpu_predict, make_runner  # noqa: E402

FEATURES = 10


def class_model(path, info, num_class, depth=4, twins=()):
    """Tree t votes for class info[t]; trees of the classes in `twins` are the same, in the same order."""
    rng = np.random.Generator(np.random.PCG64(num_class))
    grow = lambda r: synth._grow_tree(r, depth, lambda d, s: 0.8, lambda: (r.integers(0, FEATURES), r.normal()), lambda: r.normal(0.0, 0.1))
    seen, trees = {}, []
    for c in info:
        seen[c] = seen.get(c, -1) + 1
        trees.append(grow(np.random.Generator(np.random.PCG64([7, seen[c]])) if c in twins else rng))
    synth.write_xgboost_json(path, trees, FEATURES, objective="multi:softmax", num_class=num_class, tree_info=list(info))
    return str(path)


def check(runner, path, x):
    forest = model_io.load_xgboost_json(path)
    assert " ownClasses=1" in runner.describe_plan(), runner.describe_plan()
    np.testing.assert_array_equal(gpu_leaf_ids(runner, x), cpu_oracle.leaf_ids(forest, x))
    rows, classes = len(x), forest.num_classes
    dx = torch.from_numpy(x).cuda()
    ids = torch.full((rows,), -1, dtype=torch.int8, device="cuda")
    margins = torch.full((rows, classes), -1.0, device="cuda")
    torch.cuda.synchronize()
    runner.run_device_multiclass(dx.data_ptr(), rows, ids.data_ptr(), margins.data_ptr(), None)
    sums = cpu_oracle.predict(forest, x)[1]
    sums = np.where(np.isin(np.arange(classes), forest.class_id)[None, :], sums, forest.initial_value).astype(np.float32)
    expected = cpu_oracle.argmax_generated(sums)  # (of equal sums the larger class id)
    np.testing.assert_array_equal(ids.cpu().numpy(), expected)
    np.testing.assert_array_equal(gpu_predict(runner, x), expected)
    np.testing.assert_allclose(margins.cpu().numpy(), sums, rtol=RTOL_SUM, atol=1e-7)


@pytest.mark.parametrize("classes,threads", [(2, 2), (2, 8), (3, 4), (4, 4), (5, 4), (7, 4), (8, 4), (9, 8), (12, 2), (12, 16), (16, 16), (40, 16)])
@pytest.mark.parametrize("group,slices", [(16384, 1), (65536, 1), (16384, 3)])
def test_own_classes_match_the_oracle(tmp_path, classes, threads, group, slices):
    path = class_model(tmp_path / "m.json", [t % classes for t in range(5 * classes + 1)], classes)
    runner = make_runner(path, 1000)
    rows = 64 if threads == 16 else 128
    runner.set_plan(rows, threads, 2, group, slices)
    check(runner, path, np.random.Generator(np.random.PCG64(3)).normal(size=(1000, FEATURES)).astype(np.float32))


def test_classes_without_trees_and_unequal_classes(tmp_path):
    info = [0] * 3 + [3] * 9 + [4] * 2 + [5] * 7 + [8]     # 1, 2, 6, 7 and 9 have none
    path = class_model(tmp_path / "m.json", info, 10)
    runner = make_runner(path, 500)
    for threads in (2, 4, 8):                 
        runner.set_plan(128, threads, 4, 32768, 1)
        check(runner, path, np.random.Generator(np.random.PCG64(4)).normal(size=(500, FEATURES)).astype(np.float32))


def test_equal_sums_go_to_the_larger_class(tmp_path):
    path = class_model(tmp_path / "m.json", [t % 8 for t in range(48)], 8, twins=(1, 2, 6))
    runner = make_runner(path, 3000)
    runner.set_plan(256, 4, 4, 32768, 1)
    x = np.random.Generator(np.random.PCG64(5)).normal(size=(3000, FEATURES)).astype(np.float32)
    check(runner, path, x)
    pred = gpu_predict(runner, x)
    assert (pred == 6).any() and not np.isin(pred, (1, 2)).any()


def test_even_split_of_own_classes(tmp_path):
    path = class_model(tmp_path / "m.json", [t % 8 for t in range(400)], 8, depth=6)
    rows = 256 * 300 + 7
    runner = make_runner(path, rows)
    assert "batchKernel=rows_lds_split" in runner.describe_plan(), runner.describe_plan()
    assert " ownClasses=1" in runner.describe_plan()
    x = np.random.Generator(np.random.PCG64(6)).normal(size=(rows, FEATURES)).astype(np.float32)
    forest = model_io.load_xgboost_json(path)
    dx = torch.from_numpy(x).cuda()
    margins = torch.zeros((rows, 8), device="cuda")
    ids = torch.zeros(rows, dtype=torch.int8, device="cuda")
    torch.cuda.synchronize()
    runner.run_device_multiclass(dx.data_ptr(), rows, ids.data_ptr(), margins.data_ptr(), None)
    pred, sums = cpu_oracle.predict(forest, x)
    np.testing.assert_array_equal(ids.cpu().numpy().astype(np.float32), pred)
    np.testing.assert_allclose(margins.cpu().numpy(), sums, rtol=RTOL_SUM, atol=1e-7)


def test_a_base_score_that_is_no_number(tmp_path):
    """Every sum is NaN: the class the running rule ends with is the last one, as without classes of the tree threads' own."""
    path = class_model(tmp_path / "m.json", [t % 7 for t in range(35)], 7)
    text = open(path).read()
    assert text.count('"base_score"') == 1
    start = text.index('"', text.index(":", text.index('"base_score"'))) + 1
    open(path, "w").write(text[:start] + "nan" + text[text.index('"', start):])
    x = np.random.Generator(np.random.PCG64(8)).normal(size=(500, FEATURES)).astype(np.float32)
    for threads, own in ((1, 0), (4, 1), (2, 1)):
        runner = make_runner(path, 500)
        runner.set_plan(128, threads, 2, 32768, 1)
        assert " ownClasses=%d" % own in runner.describe_plan()
        np.testing.assert_array_equal(gpu_predict(runner, x), np.full(500, 6))
