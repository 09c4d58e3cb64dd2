"""Wide rows on one-byte ranks, bundles of trees streamed by each wave: feature counts at both ends of the form's range,
up to 254 thresholds per feature, trees from one leaf to 255 splits, values on thresholds, non-finite rows, ragged batches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle, model_io  # noqa: E402
from treebeard_amd import synth  # noqa: E402

from test_gpu_few_rows import close, limit_of  # noqa: E402
from test_gpu_parity import gpu_predict, make_runner  # noqa: E402


@pytest.mark.parametrize("features,trees,depth,split,levels", [(600, 3, 8, 1.0, 254), (600, 160, 7, 0.8, 254), (1100, 61, 6, 0.9, 127),
                                                               (2000, 700, 5, 0.8, 31), (2047, 120, 8, 0.75, 254)])
def test_streamed_bundles_match_the_oracle(tmp_path, features, trees, depth, split, levels):
    rng = np.random.Generator(np.random.PCG64(features + trees))
    grid = np.sort(rng.standard_normal(levels)).astype(np.float32)

    def draw_split():
        return rng.integers(0, features), grid[rng.integers(0, levels)]
    forest_trees = [synth._grow_tree(rng, depth if t % 7 else t // 7 % 3, lambda d, s: split, draw_split, lambda: rng.normal(), force_root=t % 7 > 0)
                    for t in range(trees)]
    path = str(tmp_path / "wide.json")
    synth.write_xgboost_json(path, forest_trees, features)
    forest = model_io.load_xgboost_json(path)
    runner = make_runner(path, 20000)
    assert "quantizedRows=1" in runner.describe_plan()
    few = limit_of(runner)
    rows = max(few, 2000) + 701
    x = rng.standard_normal((rows, features), dtype=np.float32)
    x[::3] = grid[rng.integers(0, levels, (len(x[::3]), features))]
    x[rows - 1, :] = np.nan
    x[rows - 2, :] = np.inf
    x[rows - 3, ::2] = -np.inf
    expected = cpu_oracle.predict(forest, x)[0]
    for count in (rows, rows - 32, few + 1, few + 33):
        close(forest, gpu_predict(runner, x[rows - count:]), expected[rows - count:])
    out = torch.zeros(rows, device="cuda")
    dx = torch.from_numpy(x).cuda()
    stream = torch.cuda.current_stream()
    for call in (runner.run_device_async, runner.run_device_noalloc):
        out.zero_()
        call(dx.data_ptr(), out.data_ptr(), rows, stream.cuda_stream)
        stream.synchronize()
        close(forest, out.cpu().numpy(), expected)


@pytest.mark.parametrize("trees", [3, 150])
def test_workgroups_that_take_several_row_blocks(tmp_path, trees):
    """More blocks of 32 rows than compute units: two and three per workgroup, the last of some only; three trees leave most
    waves without a bundle, 150 leave them unequal numbers."""
    rng = np.random.Generator(np.random.PCG64(trees))
    features, levels = 600, 31
    grid = np.sort(rng.standard_normal(levels)).astype(np.float32)
    forest_trees = [synth._grow_tree(rng, 6, lambda d, s: 0.9, lambda: (rng.integers(0, features), grid[rng.integers(0, levels)]), rng.normal)
                    for _ in range(trees)]
    path = str(tmp_path / "wide.json")
    synth.write_xgboost_json(path, forest_trees, features)
    forest = model_io.load_xgboost_json(path)
    runner = make_runner(path, 20000)
    assert "quantizedRows=1" in runner.describe_plan()
    x = rng.standard_normal((2 * 8192 + 4 * 32 + 5, features), dtype=np.float32)
    expected = cpu_oracle.predict(forest, x)[0]
    counts = [c for c in (8192, 8192 + 1, 8192 + 700, len(x)) if c > limit_of(runner)]
    assert counts
    for count in counts:
        close(forest, gpu_predict(runner, x[:count]), expected[:count])


@pytest.mark.parametrize("depths", [[0] * 19 + [1] * 3 + [8], [1] * 9, [0] * 17 + [2], [8] * 5 + [0, 1, 2], [0] * 3 + [3] * 30])
def test_bundles_of_the_smallest_trees(tmp_path, depths):
    """Bundles that are walked no level, one and two: their trees' roots stand in the bundle's head, those that split only there."""
    rng = np.random.Generator(np.random.PCG64(len(depths)))
    features, levels = 600, 60
    grid = np.sort(rng.standard_normal(levels)).astype(np.float32)
    forest_trees = [synth._grow_tree(rng, depth, lambda d, s: 1.0, lambda: (rng.integers(0, features), grid[rng.integers(0, levels)]),
                                     rng.normal, force_root=depth > 0) for depth in depths]
    path = str(tmp_path / "small.json")
    synth.write_xgboost_json(path, forest_trees, features)
    forest = model_io.load_xgboost_json(path)
    runner = make_runner(path, 20000)
    rows = max(limit_of(runner), 2000) + 33
    x = rng.standard_normal((rows, features), dtype=np.float32)
    x[::3] = grid[rng.integers(0, levels, (len(x[::3]), features))]
    x[rows - 1, :] = np.nan
    x[rows - 2, :] = np.inf
    close(forest, gpu_predict(runner, x), cpu_oracle.predict(forest, x)[0])
