"""A step that is refused leaves every export of the live meetings as it was: keys, fields and units of the last step that
was completed, for steps from positions and from replayed units, and the next step goes on from there."""
import numpy as np
import pytest

import oracle_lib as O
from stcdb_amd import Pipeline, gen_params, map_box, pipeline_config
from stcdb_amd._lib import STC_E_INPUT, StcError

pytestmark = pytest.mark.gpu


def exports(p):
    return [p.step_meeting_units().view(np.uint8), p.pairs(), *(a.view(np.uint8) for a in p.active())]


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("dynamic", [0, 1])
def test_points_outside_the_map(dynamic):
    n = 2000
    gp = gen_params(n, 20, seed=1)
    box = map_box(gp)
    lo, hi = np.array(box[0]), np.array(box[1])
    rng = np.random.default_rng(4)
    cfg = pipeline_config(n, 15.0, 2, grid_capacity=30, kv_restriction=1 << 20, keep_pairs=1, dynamic_schema=dynamic)
    gpu, orc = Pipeline(cfg, box), O.Oracle(cfg, box)
    xy = rng.uniform(lo + 1e-3 * (hi - lo), hi - 1e-3 * (hi - lo), (n, 2))
    for t in range(3):
        gpu.step(xy, t)
        orc.step(xy, t)
        before = exports(gpu)
        bad = rng.uniform(lo + 1e-3 * (hi - lo), hi - 1e-3 * (hi - lo), (n, 2))  # other places, one of them outside
        bad[n // 2] = hi + 1.0
        with pytest.raises(StcError) as e:
            gpu.step(bad, t + 1)
        assert e.value.code == STC_E_INPUT
        assert same(exports(gpu), before), t
        ok, os_, oe, om = orc.active()
        assert len(ok) and np.array_equal(before[1], ok)
        assert np.array_equal(before[0].reshape(-1, 32)[:, 16:], units_boxes(ok, xy))
        xy = xy + rng.normal(0, 3e-5, xy.shape)
        xy = np.clip(xy, lo + 1e-3 * (hi - lo), hi - 1e-3 * (hi - lo))
    gpu.close()
    orc.close()


def units_boxes(keys, xy):
    f = xy.astype(np.float32)
    a, b = f[(keys >> np.uint64(32)).astype(np.int64)], f[(keys & np.uint64(0xFFFFFFFF)).astype(np.int64)]
    return np.concatenate([np.minimum(a, b), np.maximum(a, b)], axis=1).view(np.uint8)


def test_units_that_name_no_pair():
    n = 2000
    gp = gen_params(n, 20, seed=1)
    box = map_box(gp)
    lo, hi = np.array(box[0]), np.array(box[1])
    rng = np.random.default_rng(5)
    cfg = pipeline_config(n, 15.0, 2, grid_capacity=30, kv_restriction=1 << 20, keep_pairs=1)
    src, rep = Pipeline(cfg, box), Pipeline(cfg, box)
    for t in range(3):
        src.step(rng.uniform(lo + 1e-3 * (hi - lo), hi - 1e-3 * (hi - lo), (n, 2)), t)
        units = src.step_meeting_units()
        rep.step_meetings(units, t)
        before = exports(rep)
        assert np.array_equal(before[0], units.view(np.uint8))
        bad = units[::-1][: len(units) // 2 + 1].copy()
        bad["mbr"] += 1.0
        for key in (np.uint64(0), units["key"][len(units) - 1]):  # no two objects; a pair named twice
            bad["key"][-1] = key
            with pytest.raises(StcError) as e:
                rep.step_meetings(bad, t + 1)
            assert e.value.code == STC_E_INPUT
            assert same(exports(rep), before), t
    src.close()
    rep.close()
