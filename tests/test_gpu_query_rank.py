"""The order of a batch's hits at the edges of how they are sorted: by the host, by ranks in tiles of 256, by radix. A
capacity below the number of hits stores as many of them, whichever, in order: each is one of the oracle's."""
import numpy as np
import pytest

from test_gpu_query_sort import ranges, state

pytestmark = pytest.mark.gpu


def test_capped_hits_are_the_oracles_in_order():
    w, gpu, orc = state(0)
    q = ranges(w, 5, 0, 1.0)
    oh, oc = orc.query(q)
    words = np.ascontiguousarray(oh).view(np.uint64).reshape(-1, 7)
    want = {r.tobytes(): k for k, r in enumerate(words)}
    assert len(oh) > 16385 and len(want) == len(oh)
    for cap in (1, 2, 255, 256, 257, 511, 512, 513, 4095, 16383, 16384, 16385):
        print(f"[query rank] cap {cap} of {len(oh)}", flush=True)
        gh, gc = gpu.query(q, cap=cap)
        assert len(gh) == cap and np.array_equal(gc, oc)
        at = [want[r.tobytes()] for r in np.ascontiguousarray(gh).view(np.uint64).reshape(-1, 7)]
        assert all(x < y for x, y in zip(at, at[1:])), cap
    gpu.close()
    orc.close()
