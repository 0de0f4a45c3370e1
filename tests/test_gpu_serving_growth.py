"""Query batches while the stepping thread's arrays grow: the memtable past its first room (and past it within one step,
so that the merge runs again), the meeting arrays of a crowd that forms, with the flush inside the step and beside it.
Every batch is answered again by a second context at the state that it saw: counts and hits are the same, bit for bit."""
import threading

import numpy as np
import pytest

import oracle_lib as O
from stcdb_amd import HostTrace, Pipeline, workload
from stcdb_amd.engine import HIT_DTYPE
from test_gpu_serving import random_queries

pytestmark = pytest.mark.gpu


def serve(cfg, ref_cfg, box, frames, seed, tag):
    n, rng = cfg["num_objects"], np.random.default_rng(seed)
    gpu = Pipeline(cfg, box)
    for t in range(3):
        gpu.step(frames[t], t)
    errors, done, grown = [], threading.Event(), []

    def ingest():
        try:
            for t in range(3, len(frames)):
                grown.append(gpu.step(frames[t], t))
        except Exception as e:
            errors.append(e)
        finally:
            done.set()

    th = threading.Thread(target=ingest)
    buf = np.zeros(1 << 21, dtype=HIT_DTYPE)
    recorded, seen = [], 2
    print(f"[growth {tag}] serving while {len(frames) - 3} steps run", flush=True)
    th.start()
    while not done.is_set() or not recorded:
        q = random_queries(rng, n, box, seen + 1, int(rng.integers(1, 9)), count_ranges=True)
        hits, counts, seen = gpu.query_at(q, buf)
        recorded.append((seen, q, hits.copy(), counts.copy()))
    th.join()
    gpu.close()
    assert not errors, errors
    ref, orc = Pipeline(ref_cfg, box), O.Oracle(ref_cfg, box)
    checked = 0
    for t in range(len(frames)):
        g, o = ref.step(frames[t], t), orc.step(frames[t], t)
        assert g["active_meetings"] == o["active"] and g["expired"] == o["expired"], (tag, t)
        batches = [r for r in recorded if r[0] == t]
        for _, q, hits, counts in batches[:40] + batches[-10:]:
            h, c = ref.query(q)
            assert np.array_equal(c, counts), (tag, t)
            assert np.array_equal(h.view(np.uint8), hits.view(np.uint8)), (tag, t)
            checked += len(h)
    print(f"[growth {tag}] {len(recorded)} batches over {len(set(r[0] for r in recorded))} states, {checked} hits equal", flush=True)
    ref.close()
    orc.close()
    return grown


def crowd(n, steps, shrink):
    """a walk whose objects are drawn together, a little more at every step"""
    w = workload("c1", num_objects=n, min_meet_time=1, kv_restriction=140_000, reach_distance=12.0, device_runs=1)
    frames = [xy.copy() for _, xy in HostTrace(w["gen"]).steps(steps)]
    centre = (np.array(w["box"][0]) + np.array(w["box"][1])) / 2
    return w, [centre + (xy - centre) * max(shrink ** t, 0.02) for t, xy in enumerate(frames)]


@pytest.mark.parametrize("flush", ["none", "sync", "async"])
def test_crowd_forms(flush):
    w, frames = crowd(30000, 26, 0.86)
    ref = dict(w["cfg"], kv_restriction=140_000 if flush == "none" else 2000)
    out = serve(dict(ref, async_flush=int(flush == "async")), ref, w["box"], frames, 3, f"crowd {flush}")
    live = [g["active_meetings"] for g in out]
    assert max(live) > 20 * live[0]  # the arrays have grown, some of them several times
    if flush == "none":
        assert 100_000 < out[-1]["kv_count"] < 140_000  # the first room, for 210,000, had to keep 131,074 free
    else:
        assert sum(g["flushed"] for g in out) > 10


def test_more_records_in_a_step_than_room():
    """a crowd that goes apart at once: more meetings end in a step than the memtable has room for"""
    w, frames = crowd(30000, 20, 0.8)
    apart = HostTrace(dict(w["gen"], seed=99))
    for t, xy in apart.steps(3):
        frames.append(xy.copy())
    out = serve(w["cfg"], w["cfg"], w["box"], frames, 5, "apart")
    k = next(i for i, g in enumerate(out) if i and g["active_meetings"] < out[i - 1]["active_meetings"] / 4)
    before = out[k - 1]["kv_count"]
    print(f"[growth apart] {out[k]['expired']} meetings ended at once, {before} records before", flush=True)
    assert out[k]["kv_count"] > 3 * (before + 2 * 131072)  # more than any room the step could have started with
