"""Batches whose tables are longer than the pinned memory that they go through (cell lists of map-wide boxes, many ids,
many candidates in the runs): the counts and hits of the same queries asked in small batches."""
import ctypes as C

import numpy as np
import pytest

from stcdb_amd import HostTrace, Pipeline, workload
from stcdb_amd._lib import STC_E_CAPACITY
from stcdb_amd.engine import HIT_DTYPE, Q_OID, Q_RANGE, QF_COUNT, QUERY_DTYPE
from test_oracle_query import make_queries
import oracle_lib as O

pytestmark = pytest.mark.gpu


def test_long_tables():
    w = workload("c1", num_objects=2500, kv_restriction=400, min_meet_time=2, device_runs=1, reach_distance=12.0)
    w["gen"].update(n_hotspots=2, hotspot_frac=0.8, hotspot_sigma=120.0)
    gpu, orc = Pipeline(w["cfg"], w["box"]), O.Oracle(w["cfg"], w["box"])
    for t, xy in HostTrace(w["gen"]).steps(12):
        gpu.step(xy, t)
        orc.step(xy, t)
    assert gpu.num_runs() >= 2
    rng = np.random.default_rng(3)
    few = make_queries(orc, w, rng, 60)
    lo, hi = np.array(w["box"][0]), np.array(w["box"][1])
    wide = few["kind"] == Q_RANGE
    few["box"][wide] = np.concatenate([lo, hi])
    few["box"][wide, :2] -= rng.random((wide.sum(), 2)) * 1e-3
    few["flags"] = np.where(wide, QF_COUNT, 0)
    few["t1"][wide] = rng.integers(2, 12, wide.sum())
    one = [gpu.query(few[i:i + 1]) for i in range(len(few))]
    many = np.concatenate([few[wide]] * 60 + [few[~wide]] * 3)  # some 1,300 map-wide boxes: 21 MB of cell lists
    assert wide.sum() * 60 * 64 * 64 * 4 > 2 * (8 << 20)
    print(f"[tables] {len(many)} queries, {wide.sum() * 60} map-wide boxes", flush=True)
    for _ in range(2):
        hits, counts = gpu.query(many)
        at = np.concatenate([np.flatnonzero(wide)] * 60 + [np.flatnonzero(~wide)] * 3)
        assert np.array_equal(counts, np.array([one[i][1][0] for i in at]))
        for k in list(range(len(many) - 3 * int((~wide).sum()), len(many)))[::7]:
            mine = hits[hits["query"] == k].copy()
            mine["query"] = 0
            assert np.array_equal(mine.view(np.uint8), one[at[k]][0].view(np.uint8))
    ids = np.zeros(200_000, dtype=few.dtype)  # 20 MB of ids and hash
    ids["kind"], ids["t1"] = Q_OID, 20
    ids["oid"] = rng.permutation(200_000) % 2500 + (np.arange(200_000) >= 5000) * 10_000  # two queries an object, the rest ask for none
    hits, counts = gpu.query(ids)
    alone, _ = gpu.query(ids[:5000])
    assert len(alone) and np.array_equal(hits.view(np.uint8), alone.view(np.uint8)) and not counts[5000:].any()
    gpu.close()
    orc.close()


def test_a_batch_too_large_is_refused_whole():
    w = workload("c1", num_objects=2500, min_meet_time=2, reach_distance=12.0)
    gpu = Pipeline(w["cfg"], w["box"])
    for t, xy in HostTrace(w["gen"]).steps(4):
        gpu.step(xy, t)
    q = np.zeros(3, dtype=QUERY_DTYPE)
    q["kind"], q["t1"], q["box"] = Q_RANGE, 9, np.concatenate([w["box"][0], w["box"][1]])
    want, counts = gpu.query(q)
    hits, n = np.zeros(16, dtype=HIT_DTYPE), C.c_uint64(77)
    ptr = [a.ctypes.data_as(C.c_void_p) for a in (q, hits)]
    rc = gpu.lib.stc_query_batch(gpu.ctx, ptr[0], len(q), ptr[1], 1 << 33, C.byref(n), None)  # 480 GB of hits
    assert rc == STC_E_CAPACITY and b"admission" in gpu.lib.stc_last_error(gpu.ctx)
    assert not hits.view(np.uint8).any()
    again, counts2 = gpu.query(q)
    assert len(want) and np.array_equal(again.view(np.uint8), want.view(np.uint8)) and np.array_equal(counts, counts2)
    gpu.close()
