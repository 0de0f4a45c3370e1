"""One step of more than 2^23 objects against the oracle: the collect and place passes' largest batches and grids, with
segments of every class of the wide place pass (65 to 512 slots), short ones and longer ones."""
import numpy as np
import pytest

import oracle_lib as O
from stcdb_amd import Pipeline, gen_params, map_box, pipeline_config

pytestmark = pytest.mark.gpu


def test_more_objects_than_the_last_rule():
    n, crowd = (1 << 23) + 4099, 24000
    gp = gen_params(n, 500, seed=1)
    box = map_box(gp)
    lo, hi = np.array(box[0]), np.array(box[1])
    rng = np.random.default_rng(8)
    xy = lo + (0.001 + 0.998 * rng.random((n, 2))) * (hi - lo)
    k = rng.choice(n, crowd, replace=False)  # the crowd's ids are spread over all
    xy[k] = (lo + hi) / 2 + (hi - lo) * rng.normal(0.0, 0.0005, (crowd, 2))
    cfg = pipeline_config(n, 6.0, 2, grid_capacity=200, kv_restriction=1 << 20, keep_pairs=1)
    print(f"[large] {n} objects, oracle", flush=True)
    orc = O.Oracle(cfg, box)
    o = orc.step(xy, 0)
    want = orc.pairs()
    orc.close()
    slots = np.bincount((want >> np.uint64(32)).astype(np.int64), minlength=n)
    print(f"[large] {len(want)} pairs, longest segment {slots.max()}", flush=True)
    assert all(((slots > a) & (slots <= b)).sum() > 20 for a, b in [(0, 64), (64, 128), (128, 256), (256, 510)])
    gpu = Pipeline(cfg, box)
    g = gpu.step(xy, 0)
    assert g["leaves"] == o["leaves"] and g["cross_units"] == o["units_cross"]
    assert np.array_equal(gpu.pairs(), want)
    gpu.close()
