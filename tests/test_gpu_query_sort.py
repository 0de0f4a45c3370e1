"""Batches with many hits, GPU against the oracle: the hits are sorted on the device by packed keys (one word, two where
the times are late, none where they do not pack: then on the host), fetched in chunks; sizes around the chunk and the
host sort's limit. Object lookups in runs whose objects have no, few and more than 64 records."""
import numpy as np
import pytest

import oracle_lib as O
from stcdb_amd import HostTrace, Pipeline, workload
from stcdb_amd.engine import HIT_DTYPE, QUERY_DTYPE, Q_OID, Q_RANGE

pytestmark = pytest.mark.gpu


def state(t0, steps=24, **over):
    w = workload("c1", num_objects=2500, kv_restriction=2000, min_meet_time=2, **over)
    w["gen"].update(n_hotspots=3, hotspot_frac=0.8, hotspot_sigma=120.0)
    cfg = dict(w["cfg"], device_runs=1, start_time=t0, reach_distance=25.0)
    gpu, orc = Pipeline(cfg, w["box"]), O.Oracle(cfg, w["box"])
    for t, xy in HostTrace(w["gen"]).steps(steps):
        gpu.step(xy, t0 + t)
        orc.step(xy, t0 + t)
    return w, gpu, orc


def ranges(w, count, t0, share):
    (lo0, lo1), (hi0, hi1) = w["box"]
    q = np.zeros(count, dtype=QUERY_DTYPE)
    q["kind"], q["t0"], q["t1"] = Q_RANGE, t0, t0 + 100
    q["box"] = (lo0, lo1, lo0 + share * (hi0 - lo0), hi1)
    return q


def same(gpu, orc, q, tag):
    gh, gc = gpu.query(q)
    oh, oc = orc.query(q)
    print(f"[query sort {tag}] {len(q)} queries, {len(oh)} hits", flush=True)
    assert gh.dtype == HIT_DTYPE and np.array_equal(gc, oc), tag
    assert np.array_equal(gh.view(np.uint8), oh.view(np.uint8)), tag
    return len(oh)


@pytest.mark.parametrize("t0", [0, 1 << 22, 1 << 27])
def test_many_hits_are_sorted(t0):
    w, gpu, orc = state(t0)
    assert gpu.num_runs() >= 1
    n = same(gpu, orc, ranges(w, 1, t0, 1.0), f"t0={t0} one")
    assert n > 1024
    most = same(gpu, orc, ranges(w, 3 + 70000 // n, t0, 1.0), f"t0={t0} chunks")
    assert most > 65536
    for share in (0.02, 0.1, 0.3):
        same(gpu, orc, ranges(w, 2, t0, share), f"t0={t0} share {share}")
    gpu.close()
    orc.close()


def test_lookups_in_runs():
    w, gpu, orc = state(0, steps=40)
    assert gpu.num_runs() >= 2
    q = np.zeros(2500, dtype=QUERY_DTYPE)
    q["kind"], q["oid"], q["t1"] = Q_OID, np.arange(2500), 1000
    _, counts = orc.query(q)
    assert counts.min() == 0 and counts.max() > 64
    same(gpu, orc, q, "lookups")
    gpu.close()
    orc.close()
