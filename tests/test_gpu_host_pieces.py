"""Host batches on their way through pinned memory in pieces and parts: sizes around every boundary of the cut, pageable and
pinned rows at odd addresses, floats and class ids, more pieces than there are buffers - the results of one device call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from treebeard_amd import synth  # noqa: E402

from test_gpu_parity import make_runner  # noqa: E402

MB = 1 << 20


@pytest.mark.parametrize("features,classes", [(3, 0), (28, 0), (28, 8), (2000, 0), (5003, 0)])
def test_pieces_give_the_results_of_one_device_call(tmp_path, features, classes):
    rng = np.random.Generator(np.random.PCG64(features + classes))
    trees = [synth._grow_tree(rng, 5, lambda d, s: 0.9, lambda: (rng.integers(0, features), rng.standard_normal()), lambda: rng.normal())
             for _ in range(40)]
    path = str(tmp_path / "host.json")
    synth.write_xgboost_json(path, trees, features, objective="multi:softmax" if classes else "reg:squarederror", num_class=classes,
                             tree_info=[t % classes for t in range(40)] if classes else None)
    row = features * 4
    runner = make_runner(path, 256)
    edges = [MB // 2, MB, 4 * MB, 16 * MB] if features < 5000 else [8 * MB, 20 * MB]
    counts = sorted({max(1, e // row + d) for e in edges for d in (-1, 0, 1, 255)} | {max(2, 45 * MB // row) | 1})
    data = rng.standard_normal(counts[-1] * features + 1).astype(np.float32)
    device = torch.from_numpy(data[1:]).cuda()
    pinned = torch.from_numpy(data).pin_memory().numpy()
    for rows in counts:
        out = torch.zeros(rows, dtype=torch.int8 if runner.result_dtype() == np.int8 else torch.float32, device="cuda")
        torch.cuda.synchronize()
        runner.run_device(device.data_ptr(), out.data_ptr(), rows)
        for host in (data, pinned):
            # (rows begin 4 bytes into the array: no copy may count on more alignment than a float's)
            np.testing.assert_array_equal(runner.run_host(host[1:1 + rows * features].reshape(rows, features)), out.cpu().numpy())


@pytest.mark.parametrize("rows", [65535, 98304, 98305, 131071, 300001])
@pytest.mark.parametrize("k", [2, 3])
def test_pieces_of_runners_compiled_for_large_batches(synth_model, k, rows):
    """Plans of one tree slice ask for pieces that fill the chip: one piece, three and more, pageable and pinned."""
    runner = make_runner(synth_model(k), 1 << 20)
    x = synth.CONFIGS[k].batch_rows(rows, seed_offset=7)
    device = torch.from_numpy(x).cuda()
    out = torch.zeros(rows, dtype=torch.int8 if runner.result_dtype() == np.int8 else torch.float32, device="cuda")
    torch.cuda.synchronize()
    runner.run_device(device.data_ptr(), out.data_ptr(), rows)
    for host in (x, torch.from_numpy(x).pin_memory().numpy()):
        # (a short piece is split between blocks, which adds its sums in another order)
        got, expected = runner.run_host(host), out.cpu().numpy()
        np.testing.assert_array_equal(got, expected) if got.dtype == np.int8 else np.testing.assert_allclose(got, expected, rtol=0, atol=1e-6)
