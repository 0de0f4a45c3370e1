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
int failed = 0, host_calls = 0;
int shim_init(const char *hip) {
    void *h = dlopen(hip, RTLD_LAZY);
    real_host = (int (*)(void **, size_t, unsigned))dlsym(h, "hipHostMalloc");
    real_dev = (int (*)(void **, size_t))dlsym(h, "hipMalloc");
    return real_host && real_dev;
}
int hipHostMalloc(void **p, size_t n, unsigned f) {
    host_calls++;
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


FLUSHES = r"""
import test_gpu_compact as T
w = workload("c1", num_objects=3000, kv_restriction=600, min_meet_time=2, max_meet_time=%d, ctf_count=16, reach_distance=15.0,
             keep_pairs=3, device_runs=%d, async_flush=%d)
w["gen"].update(n_hotspots=2, hotspot_frac=0.5, hotspot_sigma=300.0)
gpu, orc = Pipeline(w["cfg"], w["box"]), O.Oracle(dict(w["cfg"], async_flush=0), w["box"])

class Valid:
    # the packed keys that a run has: none of a CTF flagged as wider than a key can be, and those of records in CTFs alone
    # (an object that is oversize by the duration of a meeting is counted in its CTF too, as in the reference)
    def __init__(self, p):
        self.p, self.num_runs = p, p.num_runs
    def run(self, i):
        r = self.p.run(i)
        m, at, left, out = r["ctfs"], 0, r["info"]["kv_count"], []
        for cap, bits in zip(m["kv_capacity"].astype(int), m["key_bit"].astype(int)):
            if bits <= 128:
                out.append(r["key_bytes"][at:at + min(cap, left) * (bits // 8)])
            at += cap * (bits // 8)
            left = max(left - cap, 0)
        return dict(r, key_bytes=np.concatenate(out))

def same_runs(tag):
    T.same_runs(Valid(gpu), Valid(orc), tag)
frames = [xy.copy() for _, xy in HostTrace(w["gen"]).steps(30)]
flushes = 0

def refused(f, what):
    try:
        f()
    except L.StcError as e:
        assert what in str(e), e
        return True
    raise SystemExit("not refused")

def history():
    q = np.zeros(3000, dtype=QUERY_DTYPE)
    q["kind"], q["t1"], q["oid"] = Q_OID, 1000, np.arange(3000)
    out = []
    for p in (gpu, orc):
        h = p.query(q)[0]
        out.append(np.sort(np.rec.fromarrays([h[k] for k in ("pid", "target", "start", "end")])))
    return out
"""


def test_a_flush_without_pinned_memory_is_made_again(tmp_path):
    """the same run as if nothing had failed, with objects that are oversize by the duration of a meeting"""
    child(tmp_path, FLUSHES % (5, 0, 0) + r"""
for t, xy in enumerate(frames):
    o = orc.step(xy, t)
    flushes += o["flushed"]
    if o["flushed"] and flushes in (2, 5):
        host.value = 1 << 20
        assert refused(lambda: gpu.step(xy, t), "pinned run buffer")
        host.value = NONE
    g = gpu.step(xy, t)
    assert g["flushed"] == o["flushed"], t
assert failed.value >= 2 and flushes > 6
same_runs("pinned")
assert sum(orc.run(i)["info"]["oversize_count"] for i in range(flushes)) > 0
gpu.close()
print("done")
""")


def test_a_flush_beside_the_steps_that_fails_keeps_its_records(tmp_path):
    child(tmp_path, FLUSHES % (64, 1, 1) + r"""
for t, xy in enumerate(frames):
    o = orc.step(xy, t)
    flushes += o["flushed"]
    if o["flushed"] and flushes == 2:
        gpu.num_runs()
        host.value = 1 << 20
        gpu.step(xy, t)
        assert refused(gpu.num_runs, "pinned run buffer")
        host.value = NONE
    else:
        gpu.step(xy, t)
n = gpu.num_runs()
assert failed.value == 1 and n >= flushes - 2
a, b = history()
assert len(a) > 1000 and np.array_equal(a, b)
gpu.close()
print("done")
""")


def test_a_run_without_device_memory_is_still_read(tmp_path):
    child(tmp_path, FLUSHES % (64, 1, 0) + r"""
for t, xy in enumerate(frames):
    o = orc.step(xy, t)
    flushes += o["flushed"]
    if o["flushed"] and flushes == 6:
        dev.value = 1
        assert refused(lambda: gpu.step(xy, t), "run.dev")
        dev.value = NONE
    else:
        g = gpu.step(xy, t)
        assert g["flushed"] == o["flushed"], t
    if flushes == 6 and t + 1 < len(frames) and o["flushed"]:
        break
assert flushes == 6 and failed.value >= 1
same_runs("device block")
for u in range(t + 1, len(frames)):
    gpu.step(frames[u], u)
assert gpu.num_runs() > 7
gpu.close()
print("done")
""")


def test_a_context_makes_few_pinned_blocks(tmp_path):
    """each is a quarter of a millisecond to free: one of a context's own and one of its queries', and no more for its first
    step, query and flush than the run's"""
    child(tmp_path, r"""
calls = C.c_int.in_dll(shim, "host_calls")
w = workload("c1", num_objects=3000, kv_restriction=100, min_meet_time=1, reach_distance=15.0)
w["gen"].update(n_hotspots=2, hotspot_frac=0.5, hotspot_sigma=300.0)
gpu = Pipeline(w["cfg"], w["box"])
assert calls.value <= 2, calls.value
before = calls.value
q = np.zeros(5, dtype=QUERY_DTYPE)
q["kind"], q["t1"], q["oid"] = Q_OID, 100, np.arange(5)
flushed = 0
for t, xy in HostTrace(w["gen"]).steps(6):
    flushed += gpu.step(xy, t)["flushed"]
    gpu.query(q)
assert flushed and calls.value - before <= flushed, (calls.value, flushed)
gpu.close()
print("done")
""")
