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
    (131073, 90, 5, 20, (256, 4)),                                     # more than 24 KB
    (40000, 73, 5, 50, (256, 4)), (40000, 74, 5, 50, (128, 8)),        # levels for two groups beside 256 rows and one beside 128
    (163840, 60, 4, 50, (128, 4)), (163841, 60, 4, 50, (256, 4)),      # three blocks to a unit: a round and a quarter, and more
    (300000, 59, 4, 50, (128, 4))])                                    # four
def test_block_shapes_of_small_forests_and_batches(tmp_path, rows, trees, depth, features, shape):
    rng = np.random.Generator(np.random.PCG64(rows + trees))
    grown = [synth._grow_tree(rng, depth, lambda d, s: 1.0, lambda: (rng.integers(0, features), rng.normal()), lambda: rng.normal(0.0, 0.1))
             for _ in range(trees)]
    path = str(tmp_path / "m.json")
    synth.write_xgboost_json(path, grown, features)
    runner = make_runner(path, rows)
    assert "kernel=rows_lds rowsPerBlock=%d treeThreads=%d " % shape in runner.describe_plan(), runner.describe_plan()
    assert " treeSlices=1 " in runner.describe_plan()
    check_against_oracle(runner, model_io.load_xgboost_json(path), rng.standard_normal((rows, features), dtype=np.float32))


def full_tree(rng, nodes, features):
    """A tree of an odd number of nodes, level by level as full as they go."""
    tree, at = synth.TreeArrays(), np.arange(nodes)
    inner = at * 2 + 2 < nodes
    tree.left, tree.right = np.where(inner, at * 2 + 1, -1).tolist(), np.where(inner, at * 2 + 2, -1).tolist()
    tree.parent = [synth.ROOT_PARENT] + ((at[1:] - 1) // 2).tolist()
    tree.feature = np.where(inner, rng.integers(0, features, nodes), 0).tolist()
    tree.value = np.where(inner, rng.standard_normal(nodes), rng.normal(0.0, 0.1, nodes)).astype(np.float32).tolist()
    return tree


@pytest.mark.parametrize("features,nodes,trees,rows,shape", [
    (60, 6401, 1, 1000, (256, 4)), (60, 6401, 1, 40000, (256, 4)), (40, 8001, 1, 65536, (256, 4)), (25, 8189, 2, 20000, (128, 8))])
def test_big_trees_beside_the_rows_of_small_batches(tmp_path, features, nodes, trees, rows, shape):
    """Batches of fewer row blocks than compute units beside a tree that the smaller blocks' groups do not hold, and one that they do."""
    rng = np.random.Generator(np.random.PCG64(nodes))
    path = str(tmp_path / "m.json")
    synth.write_xgboost_json(path, [full_tree(rng, nodes, features) for _ in range(trees)], features)
    runner = make_runner(path, rows)
    assert "kernel=rows_lds rowsPerBlock=%d treeThreads=%d " % shape in runner.describe_plan(), runner.describe_plan()
    check_against_oracle(runner, model_io.load_xgboost_json(path), rng.standard_normal((rows, features), dtype=np.float32))
