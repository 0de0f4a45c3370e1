"""Calls that find no memory of the kind they would take first: pinned memory (exports, query batches large and small) is
replaced by plain copies, with the same results. The allocations fail by a small library loaded before the product's, in
a process of its own; every kernel runs as ever."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static int (*real_host)(void **, size_t, unsigned), (*real_dev)(void **, size_t);
size_t fail_host_from = (size_t)-1, fail_dev_from = (size_t)-1; /* allocations of at least so many bytes fail */
int failed = 0;
int shim_init(const char *hip) {
    void *h = dlopen(hip, RTLD_LAZY);
    real_host = (int (*)(void **, size_t, unsigned))dlsym(h, "hipHostMalloc");
    real_dev = (int (*)(void **, size_t))dlsym(h, "hipMalloc");
    return real_host && real_dev;
}
int hipHostMalloc(void **p, size_t n, unsigned f) {
    if (n >= fail_host_from) { failed++; return 2; }
    return real_host(p, n, f);
}
int hipMalloc(void **p, size_t n) {
    if (n >= fail_dev_from) { failed++; return 2; }
    return real_dev(p, n);
}
"""

PRELUDE = r"""
import ctypes as C, os, sys
sys.path[:0] = [os.environ["STC_ROOT"], os.path.join(os.environ["STC_ROOT"], "tests")]
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
import numpy as np
import stcdb_amd._lib as L
L.load()
hip = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
assert shim.shim_init(hip.encode())
host, dev, failed = (C.c_size_t.in_dll(shim, n) for n in ("fail_host_from", "fail_dev_from", "failed"))
failed = C.c_int.in_dll(shim, "failed")
NONE = C.c_size_t(-1).value
import oracle_lib as O
from stcdb_amd import HostTrace, Pipeline, workload
from stcdb_amd.engine import *
from stcdb_amd.engine import QUERY_DTYPE, HIT_DTYPE
"""


def child(tmp_path, body):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(src), "-o", str(so), "-ldl"], check=True, timeout=60)
    r = subprocess.run([sys.executable, "-u", "-c", PRELUDE + body, str(so)], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, STC_ROOT=os.path.dirname(HERE)))
    print(r.stdout, flush=True)
    assert r.returncode == 0 and r.stdout.strip().endswith("done"), r.stdout + r.stderr


def test_no_pinned_memory_for_exports_and_queries(tmp_path):
    child(tmp_path, r"""
w = workload("c1", num_objects=3000, kv_restriction=400, min_meet_time=2, device_runs=1, reach_distance=15.0, keep_pairs=1)
w["gen"].update(n_hotspots=2, hotspot_frac=0.9, hotspot_sigma=60.0)
gpu, orc = Pipeline(w["cfg"], w["box"]), O.Oracle(w["cfg"], w["box"])
for t, xy in HostTrace(w["gen"]).steps(12):
    gpu.step(xy, t)
    orc.step(xy, t)
host.value = 1
before = failed.value
k, s, e, m = gpu.active()
ok, os_, oe, om = orc.active()
assert len(ok) > 16384  # more than a chunk
assert np.array_equal(k, ok) and np.array_equal(s, os_) and np.array_equal(e, oe) and np.array_equal(m, om)
assert np.array_equal(gpu.pairs(), orc.pairs())
units = gpu.step_meeting_units()
a, b = ok >> np.uint64(32), ok & np.uint64(0xFFFFFFFF)
assert np.array_equal(units["key"], (a + b) * (a + b + np.uint64(1)) // np.uint64(2) + b)
assert failed.value > before
print("exports", len(ok), flush=True)
rng = np.random.default_rng(1)
for n, kind, side in [(1, 2, 1e-3), (40, 2, 2e-3), (3, 2, 1.0), (9000, 1, 0.0)]:
    q = np.zeros(n, dtype=QUERY_DTYPE)
    q["kind"], q["t1"] = kind, 50
    q["oid"] = rng.integers(0, 3000, n)
    at = xy[rng.integers(0, 3000, n)]
    q["box"] = np.concatenate([at - side, at + side], axis=1)
    before = failed.value
    hits, counts = gpu.query(q)
    want, wc = orc.query(q)
    assert np.array_equal(counts, wc) and np.array_equal(hits.view(np.uint8), want.view(np.uint8)), (n, kind)
    print("queries", n, len(hits), failed.value - before, flush=True)
host.value = NONE
assert np.array_equal(gpu.active()[0], ok)
gpu.close()
print("done")
""")
