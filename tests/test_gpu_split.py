"""Row blocks x tree groups split evenly over the blocks of a launch, the parts added by the finalize kernel: rows around
the edges of row blocks and of rounds of blocks, tree slices, classifiers with and without sums, repeated calls (the parts
of one call lie where the last one's did)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle, model_io  # noqa: E402
from treebeard_amd import synth  # noqa: E402

from test_gpu_few_rows import close  # noqa: E402
from test_gpu_parity import ATOL_PROB, RTOL_SUM, gpu_predict, make_runner, pin_own_plan  # noqa: E402


@pytest.mark.parametrize("plan", [(64, 16, 4, 16384, 2), (64, 4, 2, 8192, 5), (128, 8, 4, 32768, 3), (256, 4, 8, 16384, 1), (256, 2, 1, 40960, 4)])
@pytest.mark.parametrize("k", [2, 3, 5])
def test_split_launches_match_the_oracle(synth_model, k, plan):
    forest = model_io.load_xgboost_json(synth_model(k))
    runner = make_runner(synth_model(k), 4096)
    if plan[0] * (forest.num_features + 1) * 4 + plan[3] + plan[0] * plan[1] * 8 > 150 * 1024:
        pytest.skip("no room for this shape")
    runner.set_plan(*plan)
    rb = plan[0]
    x = synth.CONFIGS[k].batch_rows(520 * rb + 1, seed_offset=5)
    x[0, ::2] = np.inf
    x[1, ::3] = np.nan
    sizes = [1, rb - 1, rb, rb + 1, 7 * rb + 3, 256 * rb, 256 * rb + 1, 512 * rb, 512 * rb + 1, 520 * rb + 1]
    expected = cpu_oracle.predict(forest, x, threads=8)[0]
    for rows in sizes + sizes[::-1]:
        close(forest, gpu_predict(runner, x[:rows]), expected[:rows])


@pytest.mark.parametrize("rows", [2000, 65536, 65537, 131072])
def test_sums_and_probabilities_of_a_split_classifier(synth_model, rows):
    forest = model_io.load_xgboost_json(synth_model(3))
    runner = make_runner(synth_model(3), rows)
    x = synth.CONFIGS[3].batch_rows(rows, seed_offset=6)
    pred, sums = cpu_oracle.predict(forest, x, threads=8)
    dx = torch.from_numpy(x).cuda()
    for _ in range(2):
        ids = torch.full((rows,), -1, dtype=torch.int8, device="cuda")
        margins, probabilities = (torch.full((rows, forest.num_classes), -1.0, device="cuda") for _ in range(2))
        torch.cuda.synchronize()
        runner.run_device_multiclass(dx.data_ptr(), rows, ids.data_ptr(), margins.data_ptr(), probabilities.data_ptr())
        np.testing.assert_array_equal(ids.cpu().numpy().astype(np.float32), pred)
        np.testing.assert_allclose(margins.cpu().numpy(), sums, rtol=RTOL_SUM, atol=1e-7)
        z = np.exp(sums.astype(np.float64) - sums.max(axis=1, keepdims=True))
        np.testing.assert_allclose(probabilities.cpu().numpy(), z / z.sum(axis=1, keepdims=True), rtol=0, atol=ATOL_PROB)


def test_wide_rows_split_on_rank_tiles(synth_model):
    forest = model_io.load_xgboost_json(synth_model(4))
    for batch in (3000, 64 * 257):
        runner = make_runner(synth_model(4), batch)
        x = synth.CONFIGS[4].batch_rows(batch, seed_offset=6)
        expected = cpu_oracle.predict(forest, x, threads=8)[0]
        for pin in (lambda r: None, pin_own_plan):          # streamed bundles, then the rank tiles of the plan
            pin(runner)
            for rows in (batch, batch - 1, 1000):
                close(forest, gpu_predict(runner, x[:rows]), expected[:rows])


@pytest.mark.parametrize("rows,group,slices", [(90000, 38912, 48), (131072, 51712, 20)])
def test_whole_rounds_of_many_slices_are_split_too(tmp_path, rows, group, slices):
    """352 row blocks x 48 slices make 33 whole rounds of 512 blocks, 512 x 20 make 20."""
    rng = np.random.Generator(np.random.PCG64(12))
    trees = [synth._grow_tree(rng, 9, lambda d, s: 0.9, lambda: (rng.integers(0, 20), rng.normal()), rng.normal) for _ in range(500)]
    path = str(tmp_path / "m.json")
    synth.write_xgboost_json(path, trees, 20)
    runner = make_runner(path, rows)
    runner.set_plan(256, 4, 4, group, slices)
    plan = dict(item.split("=", 1) for item in runner.describe_plan().split() if "=" in item)
    places = 256 * min(2, 163840 // (int(plan["ldsBytes"]) + 512))
    assert int(plan["treeSlices"]) == slices and (rows + 255) // 256 * slices % places == 0, plan
    assert plan["batchKernel"] == "rows_lds_split", plan
    x = rng.standard_normal((rows, 20), dtype=np.float32)
    got = gpu_predict(runner, x)
    forest = model_io.load_xgboost_json(path)
    for at in (0, 44000, rows - 2000):
        np.testing.assert_allclose(got[at:at + 2000], cpu_oracle.predict(forest, x[at:at + 2000])[0], rtol=1e-5, atol=1e-6)
