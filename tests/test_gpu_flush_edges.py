"""The flush's device passes at their edges, GPU against the oracle, every byte of every run: grids wider than a word of
the CTF bitmap (one to nine CTFs on the map, so that a row of cells is several words), CTFs of more than one key chunk
and of a record or none, more CTFs than one round of the layout pass takes, objects all oversize, and objects that just
fill, or just pass, the stretch of objects that a workgroup of the CTF pass takes."""
import pytest

from stcdb_amd import workload
from test_gpu_flush import compare_runs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ctfs,more", [(4000, 1, {}), (4000, 4, {}), (4000, 9, {"compat": 1}), (300, 1, {}),
                                         (2048, 16, {}), (2049, 16, {}), (6000, 3969, {}), (4000, 16, {"area_threshold": 1e-12}),
                                         (4000, 1, {"area_threshold": 2e-8})])
def test_flush_edges(n, ctfs, more):
    w = workload("c1", num_objects=n, reach_distance=20.0, min_meet_time=2, kv_restriction=40 if n < 1000 else 1500,
                 ctf_count=ctfs, **more)
    w["gen"].update(n_hotspots=3, hotspot_frac=0.8, hotspot_sigma=300.0)
    assert compare_runs(w, 20, f"edges-{n}-{ctfs}") >= 1
