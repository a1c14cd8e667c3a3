"""bench.py prints one JSON line that a reader takes from the end of a run's output, so no part of
it may grow with the number of chains; the per-chain values go to a file of their own."""
import json

import numpy as np

import bench


def test_per_chain_values_stay_off_the_result_line(tmp_path):
    rng = np.random.default_rng(0)
    cols = {k: rng.uniform(-1e5, 1e5, 256) for k in ("n", "beta", "S", "lndetJ", "lndetJ0", "delta_cm-1")}
    path = tmp_path / "chains.json"
    out = bench.per_chain(cols, str(path))
    assert len(json.dumps(out)) < 600 and out == bench.per_chain(cols)
    table = json.loads(path.read_text())
    for k, v in cols.items():
        assert np.allclose(table[k], v, rtol=1e-9, atol=0.0)
        assert np.allclose(out[k], [v.min(), np.median(v), v.max()], rtol=1e-9, atol=0.0)
