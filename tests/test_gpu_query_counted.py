"""Batches that store no hit (no capacity, or every query counted) take scans without a stage for them: each kind alone and
all together, over live sets of a few waves and of many, with boxes that every meeting passes and that none does."""
import numpy as np
import pytest

import oracle_lib as O
from stcdb_amd import HostTrace, Pipeline, map_box, workload
from stcdb_amd.engine import QF_COUNT
from test_gpu_query_scan import boxes
from test_oracle_query import make_queries

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,steps", [(60, 3), (2500, 12), (20000, 5)])
def test_counts_alone(n, steps):
    w = workload("c1", num_objects=n, kv_restriction=400, min_meet_time=2, device_runs=1, reach_distance=12.0, grid_capacity=20)
    w["gen"].update(n_hotspots=2, hotspot_frac=0.8, hotspot_sigma=120.0, grid_cells=12)
    w["box"] = map_box(w["gen"])
    gpu, orc = Pipeline(w["cfg"], w["box"]), O.Oracle(w["cfg"], w["box"])
    for t, xy in HostTrace(w["gen"]).steps(steps):
        gpu.step(xy, t)
        orc.step(xy, t)
    rng = np.random.default_rng(n)
    q = make_queries(orc, w, rng, 240)
    at = np.flatnonzero(q["kind"] == 2)
    q["box"][at] = boxes(rng, w["box"], len(at))
    q["t0"][at], q["t1"][at] = 0, 20
    total = 0
    for kinds in [(1,), (2,), (3,), (1, 3), (1, 2, 3)]:
        part = q[np.isin(q["kind"], kinds)]
        _, want = orc.query(part)
        hits, counts = gpu.query(part, cap=0)
        assert len(hits) == 0 and np.array_equal(counts, want), (kinds, "no capacity")
        counted = part.copy()
        counted["flags"] = QF_COUNT
        hits, counts = gpu.query(counted)
        assert len(hits) == 0 and np.array_equal(counts, want), (kinds, "counted")
        total += int(want.sum())
    print(f"[counted] {n} objects: {total} counted", flush=True)
    assert total > 0
    gpu.close()
    orc.close()
