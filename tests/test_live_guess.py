"""How much room the live search asks for, without a GPU: a first guess that is bounded, and none where it is refused."""
import ctypes

import numpy as np
import pytest

import stcdb_amd._lib as L
from stcdb_amd import Pipeline


class SearchStub:
    """stands in for the library's live search: `found` hits, and no admission for more than `room` of them"""

    def __init__(self, found, room):
        self.found, self.room, self.asked = found, room, []

    def stc_live_search(self, ctx, pids, n_pids, hits, cap, n):
        self.asked.append(cap)
        if cap > self.room:
            return L.STC_E_CAPACITY
        n._obj.value = self.found
        if cap:
            out = np.ctypeslib.as_array(ctypes.cast(hits, ctypes.POINTER(ctypes.c_uint32)), shape=(cap * 14,))
            out[: min(cap, self.found) * 14 : 14] = np.arange(min(cap, self.found))
        return 0


@pytest.mark.parametrize("pids,found,room,asked", [
    (1, 5, 1 << 40, [1032]),                          # fits the guess
    (1, 5000, 1 << 40, [1032, 5000]),                 # does not
    (5_000_000, 7, 1 << 40, [1 << 21]),               # the guess does not grow with the list without bound
    (1_000_000, 200_000, 1 << 40, [1 << 21]),
    (5_000_000, 2_100_000, 1 << 40, [1 << 21, 2_100_000]),
    (100, 20, 100, [1824, 0, 20]),                    # a guess that is refused where the hits are not
    (100, 0, 100, [1824, 0]),
])
def test_live_search_asks_for_no_more_room_than_it_needs(pids, found, room, asked):
    p = Pipeline.__new__(Pipeline)
    p.lib, p.ctx = SearchStub(found, room), ctypes.c_void_p()
    hits = p.live_search(np.zeros(pids, dtype=np.uint32))
    assert p.lib.asked == asked
    assert np.array_equal(hits["query"], np.arange(found))
