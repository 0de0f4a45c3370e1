"""What a query batch is admitted for (stc_query_table_bytes, host code of the library): all of its tables, the range
queries' cell lists first of all, counted by an independent restatement."""
import ctypes as C

import numpy as np
import pytest

import stcdb_amd._lib as L
from stcdb_amd.engine import Q_OID, Q_PAIR, Q_RANGE, QUERY_DTYPE

GRID, FINE = 64, 256


def table_bytes(q, box):
    fn = L.load()["_Z21stc_query_table_bytesPK9stc_queryjPKd"]
    fn.restype = C.c_uint64
    m = (C.c_double * 4)(*box)
    return fn(q.ctypes.data_as(C.c_void_p), C.c_uint32(len(q)), m)


def expected(q, box):
    def cells(b):
        c = [min(max(int((b[k] - box[k % 2]) / ((box[2 + k % 2] - box[k % 2]) / GRID)), 0), GRID - 1) for k in range(4)]
        return max(c[2] - c[0] + 1, 0) * max(c[3] - c[1] + 1, 0)

    ids = int((q["kind"] != Q_RANGE).sum())
    ranges = q["box"][q["kind"] == Q_RANGE]
    slots = 64
    while ids and slots < 2 * ids:
        slots *= 2
    n = len(q)
    sizes = [8 * (n + 1), QUERY_DTYPE.itemsize * n, 4 * sum(cells(b) for b in ranges), 4 * (GRID * GRID + 1) * (len(ranges) > 0)]
    sizes += [4 * slots, 4 * slots, 4 * n, 4 * ids] if ids else []
    bits = min(slots * 32, 1 << 16) if ids else 32
    sizes.append(bits // 8 + GRID * GRID // 8 + (FINE * FINE // 8 if len(ranges) else 0))
    return sum((s + 15) // 16 * 16 for s in sizes)


@pytest.mark.parametrize("ids,ranges,side", [(1, 0, 0.0), (40, 0, 0.0), (0, 1, 0.01), (300, 500, 0.3), (0, 2000, 1.0), (70000, 5, 1.0)])
def test_all_tables_are_counted(ids, ranges, side):
    rng = np.random.default_rng(ids + ranges)
    box = [116.0, 39.0, 117.5, 40.0]
    q = np.zeros(ids + ranges, dtype=QUERY_DTYPE)
    q["kind"][:ids] = np.where(rng.random(ids) < 0.5, Q_OID, Q_PAIR)
    q["kind"][ids:] = Q_RANGE
    q["oid"] = rng.integers(0, 1 << 20, len(q))
    at = rng.random((len(q), 2)) * (1 - side)
    lo, ext = np.array(box[:2]), np.array(box[2:]) - np.array(box[:2])
    q["box"] = np.concatenate([lo + at * ext, lo + (at + side) * ext], axis=1)
    if side == 1.0:
        q["box"] = box
    got, want = table_bytes(q, box), expected(q, box)
    assert abs(got - want) <= 64 * (side not in (0.0, 1.0))  # a cell more or less where a box ends on a border
    if side == 1.0:
        assert got > ranges * GRID * GRID * 4  # 16 KB a box
