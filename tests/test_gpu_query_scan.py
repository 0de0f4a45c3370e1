"""The query scans' filters and staging at their edges, GPU against the oracle, hit for hit: boxes from a point to the
whole map and beyond it, at its corners and between cells, on maps whose fine filter cells are wider and narrower than a
meeting's box; batches of one kind alone and of all; waves with more hits than they stage, and fewer stored than found."""
import numpy as np
import pytest

import oracle_lib as O
from stcdb_amd import HostTrace, Pipeline, workload
from test_gpu_query import compare
from test_oracle_query import make_queries

pytestmark = pytest.mark.gpu


def boxes(rng, box, n):
    lo, hi = np.array(box[0]), np.array(box[1])
    at = lo + rng.random((n, 2)) * (hi - lo)
    cells = (hi - lo) / 256
    at[::3] = lo + np.round((at[::3] - lo) / cells) * cells  # on the cells' borders
    half = np.exp(rng.uniform(np.log(1e-9), np.log(1.0), (n, 1))) * (hi - lo)
    b = np.concatenate([at - half, at + half], axis=1)
    b[0], b[1] = np.concatenate([lo, hi]), np.concatenate([lo - 1, hi + 1])
    b[2], b[3] = np.concatenate([lo, lo]), np.concatenate([hi, hi])
    return b


@pytest.mark.parametrize("cells", [3, 12, 100])
def test_scan_edges(cells):
    w = workload("c1", num_objects=2500, kv_restriction=400, min_meet_time=2, device_runs=1, reach_distance=12.0)
    w["gen"].update(n_hotspots=2, hotspot_frac=0.8, hotspot_sigma=120.0, grid_cells=cells)
    from stcdb_amd import map_box
    w["box"] = map_box(w["gen"])
    gpu, orc = Pipeline(w["cfg"], w["box"]), O.Oracle(w["cfg"], w["box"])
    for t, xy in HostTrace(w["gen"]).steps(12):
        gpu.step(xy, t)
        orc.step(xy, t)
    rng = np.random.default_rng(cells)
    q = make_queries(orc, w, rng, 210)
    at = np.flatnonzero(q["kind"] == 2)
    q["box"][at] = boxes(rng, w["box"], len(at))
    q["t0"][at], q["t1"][at] = 0, 20
    found = 0
    for kinds in [(1,), (2,), (3,), (1, 2, 3)]:
        found += compare(gpu, orc, q[np.isin(q["kind"], kinds)], f"cells {cells} kinds {kinds}")
    assert found > 2000
    gpu.close()
    orc.close()


@pytest.mark.parametrize("rows", [1, 1 << 14])
def test_more_hits_than_the_first_guess(rows, monkeypatch):
    """the hits of places, asked again and again: by a second call while the device's buffer is short, at once after it"""
    import stcdb_amd.engine as engine
    monkeypatch.setattr(engine, "FETCH_ROWS", rows)
    w = workload("c1", num_objects=2500, kv_restriction=400, min_meet_time=2, device_runs=1, reach_distance=12.0)
    w["gen"].update(n_hotspots=2, hotspot_frac=0.8, hotspot_sigma=120.0)
    gpu, orc = Pipeline(w["cfg"], w["box"]), O.Oracle(w["cfg"], w["box"])
    for t, xy in HostTrace(w["gen"]).steps(12):
        gpu.step(xy, t)
        orc.step(xy, t)
    q = make_queries(orc, w, np.random.default_rng(1), 3)[:1].repeat(24)
    q["kind"], q["t0"], q["t1"] = 2, 0, 20
    q["box"] = boxes(np.random.default_rng(2), w["box"], len(q))
    sizes = []
    for n in (4, 24, 24, 8, 1):
        sizes.append(compare(gpu, orc, q[:n], f"{n} places, {rows} rows"))
    assert max(sizes) > 2 * (1 << 14) and min(sizes) > 0
    into = np.zeros(5, dtype=engine.HIT_DTYPE)
    hits, _ = gpu.query(q, into=into)
    assert len(hits) == sizes[1] and np.array_equal(hits.view(np.uint8), orc.query(q)[0].view(np.uint8))
    gpu.close()
    orc.close()
