"""Leaves of the last level of a bundle's walk that stay out of the tree groups in LDS: trees of unlike depths side by side (a tree
less deep than its bundle keeps its leaves in LDS), stumps and single leaves among them, every number of chains, both ways of
staging, row tiles of byte and of word offsets, tree slices, even splits, classes that meet and classes of the tree threads' own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")

from oracle import model_io  # noqa: E402
from treebeard_amd import synth  # noqa: E402

from test_gpu_parity import check_against_oracle, make_runner  # noqa: E402


def write_model(path, features, depths, split, classes=0):
    rng = np.random.Generator(np.random.PCG64([features, len(depths), classes]))
    trees = [synth._grow_tree(rng, int(depth), lambda d, s: split, lambda: (rng.integers(0, features), rng.normal()),
                              lambda: rng.normal(0.0, 0.1), force_root=depth > 0) for depth in depths]
    kind = dict(objective="multi:softmax", num_class=classes, tree_info=[t % classes for t in range(len(trees))]) if classes else {}
    synth.write_xgboost_json(str(path), trees, features, **kind)
    return str(path)


def rows_for(features, rows):
    x = np.random.Generator(np.random.PCG64(rows)).standard_normal((rows, features), dtype=np.float32)
    x[0, ::2] = np.inf
    x[1 % rows, ::3] = np.nan
    x[2 % rows, ::2] = -np.inf
    return x


@pytest.mark.parametrize("staging", [1, 2])
@pytest.mark.parametrize("plan", [(64, 16, 1, 16384, 1), (128, 4, 2, 8192, 1), (256, 4, 4, 16384, 1), (256, 2, 8, 24576, 1), (64, 4, 4, 12288, 2)])
@pytest.mark.parametrize("features", [9, 280])
def test_trees_of_all_depths(tmp_path, features, plan, staging):
    if (features + 1) * plan[0] * 4 + plan[3] > 158 * 1024 or (features + 1) * plan[0] > 0xFFFF:
        pytest.skip("no room for this shape")
    depths = [0, 1, 1, 2, 0, 3] + [4, 5, 6, 7, 8] * 12 + [1, 2, 3]
    path = write_model(tmp_path / "m.json", features, depths, 0.93)
    runner = make_runner(path, 300)
    runner.set_plan(*plan)
    runner.set_group_staging(staging)
    assert " leavesOutside=1" in runner.describe_plan(), runner.describe_plan()
    for rows in (1, plan[0], plan[0] + 1, 2 * plan[0] + 77):
        check_against_oracle(runner, model_io.load_xgboost_json(path), rows_for(features, rows))


@pytest.mark.parametrize("depths,split,outside", [
    ([6] * 64, 1.0, True),        # two groups of whole trees, one without the last level
    ([6] * 30, 1.0, False),       # one group either way
    ([1] * 4000, 1.0, True),      # a level of two leaves: no walk but the root's
    ([8, 9] * 60, 0.8, True)])
def test_by_the_groups_it_saves(tmp_path, depths, split, outside):
    path = write_model(tmp_path / "m.json", 20, depths, split)
    runner = make_runner(path, 1 << 20)
    assert (" leavesOutside=1" in runner.describe_plan()) == outside, runner.describe_plan()
    for rows in (3000, 131072 + 255):                       # (the second: split evenly over a round of blocks)
        check_against_oracle(runner, model_io.load_xgboost_json(path), rows_for(20, rows))


@pytest.mark.parametrize("classes,trees,own,room", [(8, 200, True, 25088), (5, 451, False, 16896)])
def test_classes(tmp_path, classes, trees, own, room):
    """Tree threads with classes of their own leave their meeting place, 8 KB, to the groups."""
    depths = [6, 6, 5, 6, 3, 6, 0][:7] * (trees // 7 + 1)
    path = write_model(tmp_path / "m.json", 54, depths[:trees], 1.0, classes)
    runner = make_runner(path, 1 << 20)
    plan = runner.describe_plan()
    assert " leavesOutside=1" in plan and " ownClasses=%d " % own in plan and " groupBytes=%d " % room in plan, plan
    for rows in (2000, 66000):
        check_against_oracle(runner, model_io.load_xgboost_json(path), rows_for(54, rows))
