"""Launch shapes by rule: trees a lane walks side by side (two where a tree group holds too few for four on every tree thread),
block shapes of small forests and of batches too small for the chip; either side of each rule, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")

from oracle import model_io  # noqa: E402
from treebeard_amd import synth  # noqa: E402

from test_gpu_parity import check_against_oracle, make_runner  # noqa: E402


@pytest.mark.parametrize("classes", [0, 3])
@pytest.mark.parametrize("features,depth,expected", [(20, 6, 4), (20, 11, 2), (90, 6, 4), (90, 9, 2), (130, 5, 4), (130, 8, 2)])
def test_interleave_follows_the_trees_a_group_holds(tmp_path, features, depth, expected, classes):
    rng = np.random.Generator(np.random.PCG64(depth))
    trees = [synth._grow_tree(rng, depth, lambda d, s: 1.0, lambda: (rng.integers(0, features), rng.normal()), lambda: rng.normal(0.0, 0.1))
             for _ in range(15)]
    path = str(tmp_path / "m.json")
    kind = dict(objective="multi:softmax", num_class=classes, tree_info=[t % classes for t in range(15)]) if classes else {}
    synth.write_xgboost_json(path, trees, features, **kind)
    runner = make_runner(path, 100000)
    assert " interleave=%d " % expected in runner.describe_plan(), runner.describe_plan()
    x = rng.standard_normal((20001, features), dtype=np.float32)
    check_against_oracle(runner, model_io.load_xgboost_json(path), x)


@pytest.mark.parametrize("rows,trees,depth,features,shape", [
    (65536, 100, 7, 20, (128, 8)), (65537, 100, 7, 20, (256, 4)),      # a block of 256 rows for every one of 256 units, and one more
    (30000, 40, 4, 20, (128, 4)), (65536, 40, 4, 20, (128, 4)),        # few trees as well
    (131072, 40, 4, 20, (256, 4)), (131073, 40, 4, 20, (128, 4)),      # few trees, at most and more than a round of blocks
    (131073, 90, 5, 20, (256, 4))])                                    # more than 24 KB
def test_block_shapes_of_small_forests_and_batches(tmp_path, rows, trees, depth, features, shape):
    rng = np.random.Generator(np.random.PCG64(rows + trees))
    grown = [synth._grow_tree(rng, depth, lambda d, s: 1.0, lambda: (rng.integers(0, features), rng.normal()), lambda: rng.normal(0.0, 0.1))
             for _ in range(trees)]
    path = str(tmp_path / "m.json")
    synth.write_xgboost_json(path, grown, features)
    runner = make_runner(path, rows)
    assert "kernel=rows_lds rowsPerBlock=%d treeThreads=%d " % shape in runner.describe_plan(), runner.describe_plan()
    if "treeSlices=1 " in runner.describe_plan():
        check_against_oracle(runner, model_io.load_xgboost_json(path), rng.standard_normal((rows, features), dtype=np.float32))
