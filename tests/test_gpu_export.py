"""The exports of the live meetings (all fields, pair keys, meeting units) at the edges of their tiles and chunks, GPU
against the oracle: from none to several chunks, capacities below the count, live sets with dead buckets among them,
and the units of a replayed step."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from stcdb_amd import Pipeline, gen_params, map_box, pipeline_config
from stcdb_amd.engine import MEETING_UNIT_DTYPE

pytestmark = pytest.mark.gpu


def partial(gpu, cap):
    n = C.c_uint64()
    k, s, e = np.zeros(cap, np.uint64), np.zeros(cap, np.uint32), np.zeros(cap, np.uint32)
    m = np.zeros((cap, 4), np.float32)
    rc = gpu.lib.stc_get_active(gpu.ctx, *(a.ctypes.data_as(C.c_void_p) for a in (k, s, e, m)), cap, C.byref(n))
    assert rc == 0
    return n.value, k, s, e, m


@pytest.mark.parametrize("n,km,reach", [(300, 9.0, 3.0), (2000, 2.0, 12.0), (9000, 2.0, 20.0), (20000, 1.8, 25.0)])
def test_exports(n, km, reach):
    gp = gen_params(n, int(km * 10), seed=2)
    box = map_box(gp)
    rng = np.random.default_rng(n)
    cfg = pipeline_config(n, reach, 2, grid_capacity=30, kv_restriction=1 << 20, keep_pairs=1)
    gpu, orc, rep = Pipeline(cfg, box), O.Oracle(cfg, box), Pipeline(cfg, box)
    lo, hi = np.array(box[0]), np.array(box[1])
    lo, hi = lo + 1e-3 * (hi - lo), hi - 1e-3 * (hi - lo)  # a point on the map's high edges is an input error
    xy = rng.uniform(lo, hi, (n, 2))
    for t in range(3):
        r = gpu.step(xy, t)
        orc.step(xy, t)
        xy = np.clip(xy + rng.normal(0, 3e-5, xy.shape), lo, hi)
        gk, gs, ge, gm = gpu.active()
        ok, os_, oe, om = orc.active()
        print(f"[export {n}] step {t}: {len(ok)} live of {r['table_buckets']} buckets", flush=True)
        assert np.array_equal(gk, ok) and np.array_equal(gs, os_) and np.array_equal(ge, oe)
        assert np.array_equal(gm.view(np.uint32), om.view(np.uint32))
        assert np.array_equal(gpu.pairs(), orc.pairs())
        units = gpu.step_meeting_units()
        a, b = ok >> np.uint64(32), ok & np.uint64(0xFFFFFFFF)
        assert np.array_equal(units["key"], (a + b) * (a + b + np.uint64(1)) // np.uint64(2) + b)
        rep.step_meetings(units[rng.permutation(len(units))], t)
        again = rep.step_meeting_units()
        assert again.dtype == MEETING_UNIT_DTYPE and np.array_equal(again.view(np.uint8), units.view(np.uint8))
    for cap in {0, 1, 1023, 1024, 1025, 16384, 16385, len(ok) // 2, len(ok)}:
        if cap <= len(ok):
            m, k, s, e, mb = partial(gpu, cap)
            assert m == len(ok) and np.array_equal(k, ok[:cap]) and np.array_equal(s, os_[:cap])
            assert np.array_equal(e, oe[:cap]) and np.array_equal(mb.view(np.uint32), om[:cap].view(np.uint32))
    for p in (gpu, orc, rep):
        p.close()


def test_exports_among_dead_buckets():
    """pairs a few ulps from the reach distance, near the origin, where a coordinate's ulp is far below the guard band:
    the combinations that the host then rejects leave dead buckets"""
    n, reach, box = 3000, 10.0, [[0.0001, 0.0001], [0.0022, 0.0022]]
    rng = np.random.default_rng(1)
    a = rng.uniform(0.0002, 0.0020, (n // 2, 2))
    b = a + np.array([0.0, reach * (360.0 / (40076.0 * 1000.0))])
    for i in range(n // 2):
        for _ in range(int(rng.integers(0, 6))):
            b[i, 1] = np.nextafter(b[i, 1], np.inf if rng.random() < 0.5 else -np.inf)
    xy = np.concatenate([a, b])
    cfg = pipeline_config(n, reach, 2, grid_capacity=30, kv_restriction=1 << 20, keep_pairs=1)
    gpu, orc = Pipeline(cfg, box), O.Oracle(cfg, box)
    for t in range(2):
        r = gpu.step(xy, t)
        orc.step(xy, t)
        gk, gs, _, gm = gpu.active()
        ok, os_, _, om = orc.active()
        assert np.array_equal(gk, ok) and np.array_equal(gs, os_) and np.array_equal(gm.view(np.uint32), om.view(np.uint32))
        assert np.array_equal(gpu.pairs(), orc.pairs())
    print(f"[export dead] {len(ok)} live of {r['table_buckets']} buckets, {r['ambiguous_pairs']} in the band", flush=True)
    assert r["table_buckets"] > len(ok)
    gpu.close()
    orc.close()
