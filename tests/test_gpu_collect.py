"""The pair collect pass at the edges of its owner batches, GPU against the oracle: the three batch sizes (4 owners a
wave below 32k objects, 16 below 4M, 64 above) with object counts just past a multiple of the batch, and owners with
more sources than a wave lists (more than 126 cross units), which take a pass of their own."""
import numpy as np
import pytest

import oracle_lib as O
from stcdb_amd import Pipeline, gen_params, map_box, pipeline_config
from stcdb_amd.workloads import DPM_LAT, LAT0, LON0, dpm_lon

pytestmark = pytest.mark.gpu


def compare(cfg, box, frames, tag):
    gpu, orc = Pipeline(dict(cfg, keep_pairs=1), box), O.Oracle(dict(cfg, keep_pairs=1), box)
    for t, xy in enumerate(frames):
        print(f"[collect {tag}] n={len(xy)} step {t}", flush=True)
        g, o = gpu.step(xy, t), orc.step(xy, t)
        assert g["leaves"] == o["leaves"] and g["cross_units"] == o["units_cross"]
        assert np.array_equal(gpu.pairs(), orc.pairs()), (tag, t)
    out = dict(g, found=len(orc.pairs()))
    gpu.close()
    orc.close()
    return out


@pytest.mark.parametrize("n,km,reach,steps", [(5, 1.0, 400.0, 2), (4099, 2.0, 12.0, 2), (32767, 6.0, 9.0, 2),
                                              (32769, 6.0, 9.0, 2), (70003, 8.0, 20.0, 2), (4194305, 50.0, 4.0, 1)])
def test_batch_sizes(n, km, reach, steps):
    gp = gen_params(n, int(km * 10), seed=3)
    box = map_box(gp)
    rng = np.random.default_rng(n)
    frames = [rng.uniform(box[0], box[1], (n, 2)) for _ in range(steps)]
    cfg = pipeline_config(n, reach, 2, grid_capacity=2 if n < 100 else 60, kv_restriction=1 << 20)
    assert compare(cfg, box, frames, f"batch {n}")["found"] > 0


@pytest.mark.parametrize("side", [12, 30])
def test_owners_with_more_sources_than_a_wave_lists(side):
    """one object a leaf on a lattice of 1.5 m: hundreds of leaves within reach of each (some below the limit, at 12)"""
    n = side * side
    gp = gen_params(n, 100, seed=1)
    k = np.arange(n)
    m = np.stack([k % side, k // side], axis=1) * 1.5 + 4000.3
    rng = np.random.default_rng(side)
    frames = []
    for _ in range(2):
        xy = m + rng.uniform(-0.2, 0.2, m.shape)
        frames.append(np.stack([LON0 + xy[:, 0] * dpm_lon(LAT0), LAT0 + xy[:, 1] * DPM_LAT], axis=1)[rng.permutation(n)])
    cfg = pipeline_config(n, 30.0, 2, grid_capacity=1, kv_restriction=1 << 20)
    r = compare(cfg, map_box(gp), frames, f"lattice {side}")
    assert r["cross_units"] > 126 * n / 4
