"""The prefix sum on its own at the edges of its two levels: a tile, the most tiles whose sums a workgroup adds up itself,
and beyond them the level above, whose sums are scanned in place; out of place and in place, with the total, and with no
value touched past the end."""
import ctypes as C

import numpy as np
import pytest
import torch

import stcdb_amd._lib as L

pytestmark = pytest.mark.gpu

TILE, SUMS = 4096, 4096


@pytest.mark.parametrize("n", [1, TILE, TILE + 1, TILE * SUMS, TILE * SUMS + 1, TILE * SUMS + 3 * TILE + 77])
@pytest.mark.parametrize("in_place", [False, True])
def test_exclusive_scan(n, in_place):
    lib = L.load()
    scan = lib["_Z22stc_exclusive_scan_u32PKjPjjS1_S1_P12ihipStream_t"]
    words = lib["_Z20stc_radix_temp_wordsj"]
    words.restype = C.c_size_t
    need = words(C.c_uint32(n))
    print(f"[scan] {n} values, {need} words of scratch, in place {in_place}", flush=True)
    rng = np.random.default_rng(n)
    a = rng.integers(0, 200, n, dtype=np.uint32)  # the sum stays below 2^32
    mark = 0x5A5A5A5A
    src = torch.from_numpy(np.concatenate([a, np.full(8, mark, np.uint32)]).view(np.int32)).cuda()
    out = src if in_place else torch.full((n + 8,), mark, dtype=torch.int32, device="cuda")
    temp = torch.full((need + 8,), mark, dtype=torch.int32, device="cuda")
    total = torch.full((2,), mark, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    p = [C.c_void_p(t.data_ptr()) for t in (src, out, total, temp)]
    assert scan(p[0], p[1], C.c_uint32(n), p[2], p[3], C.c_void_p(None)) == 0
    torch.cuda.synchronize()
    got = out.cpu().numpy().view(np.uint32)
    want = np.cumsum(a, dtype=np.uint64)
    assert want[-1] < 1 << 32
    assert np.array_equal(got[:n], np.concatenate([[0], want[:-1]]).astype(np.uint32))
    assert (got[n:] == mark).all() and (temp.cpu().numpy()[need:] == mark).all()
    assert total.cpu().numpy().view(np.uint32).tolist() == [int(want[-1]), mark]
    if not in_place:
        assert np.array_equal(src.cpu().numpy().view(np.uint32)[:n], a)
