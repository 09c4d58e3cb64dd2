"""Rows on their way into local memory: feature counts around the pieces and lane splits of the copy, ragged last blocks,
rows that begin 4 bytes off a 16-byte boundary, the last row at the very end of its allocation."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle, model_io  # noqa: E402
from treebeard_amd import synth  # noqa: E402

from test_gpu_few_rows import close  # noqa: E402
from test_gpu_parity import make_runner  # noqa: E402


@pytest.mark.parametrize("features", [1, 3, 4, 5, 7, 12, 13, 16, 17, 33, 63, 65, 130, 255, 301])
def test_every_value_of_every_row_arrives(tmp_path, features):
    rng = np.random.Generator(np.random.PCG64(features))
    # every feature decides in some tree
    trees = [synth._grow_tree(rng, 2, lambda d, s: 1.0, lambda: ((t * 3 + rng.integers(0, 3)) % features, rng.standard_normal()),
                              lambda: rng.normal()) for t in range(max(20, features // 2))]
    path = str(tmp_path / "stage.json")
    synth.write_xgboost_json(path, trees, features)
    forest = model_io.load_xgboost_json(path)
    x = rng.standard_normal((4129, features), dtype=np.float32)
    expected = cpu_oracle.predict(forest, x)[0]
    runner = make_runner(path, 4096)
    dx = torch.from_numpy(np.concatenate([np.zeros(1, np.float32), x.ravel()])).cuda()
    for rows_per_block, tree_threads in ((64, 16), (128, 6), (256, 4)):
        if rows_per_block * features * 4 > 100 * 1024:                                # (does not fit a block's local memory)
            continue
        runner.set_plan(rows_per_block, tree_threads, 2)
        for rows in (1, 63, 65, 257, 4129):
            out = torch.zeros(rows, device="cuda")
            torch.cuda.synchronize()
            runner.run_device(dx.data_ptr() + 4 + 4 * features * (4129 - rows), out.data_ptr(), rows)
            close(forest, out.cpu().numpy(), expected[4129 - rows:])
