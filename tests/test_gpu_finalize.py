"""Class ids, sums and softmax of batches around the sizes at which a block of the finalize kernel takes more rows than a sum per
lane, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle, model_io  # noqa: E402
from treebeard_amd import synth  # noqa: E402

from test_gpu_own_classes import FEATURES, class_model  # noqa: E402
from test_gpu_parity import RTOL_SUM, check_against_oracle, make_runner  # noqa: E402


# blocks of a sum per lane and of twice as many rows, either side of the line; the largest (256 rows, 2048 sums); blocks of 8 rows and more
@pytest.mark.parametrize("classes,rows", [(2, 131071), (2, 196607), (2, 196608), (2, 262145), (5, 78847), (5, 78848), (5, 300001), (12, 32767), (12, 32768),
                                          (12, 200003), (16, 131073), (100, 11000), (100, 20481)])
def test_blocks_of_more_rows_than_a_sum_per_lane(tmp_path, classes, rows):
    path = class_model(tmp_path / "m.json", [t % classes for t in range(2 * classes + 1)], classes, depth=3)
    runner = make_runner(path, rows)
    x = np.random.Generator(np.random.PCG64(rows)).standard_normal((rows, FEATURES), dtype=np.float32)
    dx = torch.from_numpy(x).cuda()
    ids = torch.full((rows,), -1, dtype=torch.int8, device="cuda")
    margins = torch.full((rows, classes), -1.0, device="cuda")
    probabilities = torch.full((rows, classes), -1.0, device="cuda")
    torch.cuda.synchronize()
    runner.run_device_multiclass(dx.data_ptr(), rows, ids.data_ptr(), margins.data_ptr(), probabilities.data_ptr())
    sums = cpu_oracle.predict(model_io.load_xgboost_json(path), x)[1]
    np.testing.assert_allclose(margins.cpu().numpy(), sums, rtol=RTOL_SUM, atol=1e-7)
    got = margins.cpu().numpy()
    np.testing.assert_array_equal(ids.cpu().numpy(), cpu_oracle.argmax_generated(got))
    wide = got.astype(np.float64)
    wide = np.exp(wide - wide.max(axis=1, keepdims=True))
    # (the sums are rounded to 32 bits in `got`, half a unit in the last place of values below 2: 1.2e-7 in the exponent)
    np.testing.assert_allclose(probabilities.cpu().numpy(), wide / wide.sum(axis=1, keepdims=True), rtol=1e-6, atol=1e-9)


@pytest.mark.parametrize("slices", [5, 6, 7, 8, 9])
def test_plain_sums_of_several_slices(synth_model, slices):
    """A lane per row, four waves that share the slices, eight."""
    for rows in (1, 64, 2047, 65537):
        runner = make_runner(synth_model(2), rows)
        runner.set_plan(64, 2, 2, 8192, slices)
        assert " treeSlices=%d " % slices in runner.describe_plan()
        check_against_oracle(runner, model_io.load_xgboost_json(synth_model(2)), synth.CONFIGS[2].batch_rows(rows, seed_offset=3))
