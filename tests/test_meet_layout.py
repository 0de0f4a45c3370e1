"""Where a step's meetings lie (stcdb_amd/csrc/stc_table.h): in blocks without a gap, a block's MBRs, keys and starts in rows
of whole 128-byte lines, no two entries over each other. The header alone is compiled, with the host's compiler."""
import os
import subprocess

import numpy as np

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stcdb_amd", "csrc")

PROGRAM = r"""
#include "stc_table.h"
#include <cstdio>
int main() {
    printf("%u %u\n", MEET_BLOCK, MEET_BLOCK_BYTES);
    for (uint64_t i = 0; i < 3 * MEET_BLOCK; i++)
        printf("%llu %llu %llu\n", (unsigned long long)meet_mbr_at(i), (unsigned long long)meet_key_at(i), (unsigned long long)meet_start_at(i));
    const uint64_t far = 4294967294ull; /* the last meeting that a step can have */
    printf("%llu %llu %llu\n", (unsigned long long)meet_mbr_at(far), (unsigned long long)meet_key_at(far), (unsigned long long)meet_start_at(far));
    return 0;
}
"""


def test_blocks_of_whole_lines(tmp_path):
    src, exe = tmp_path / "layout.cpp", tmp_path / "layout"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True, timeout=120)
    rows = [tuple(map(int, line.split())) for line in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.splitlines()]
    (block, size), at, last = rows[0], rows[1:-1], rows[-1]
    assert size == 28 * block and size % 128 == 0
    used = np.zeros(3 * size, dtype=np.int64)
    for entry in at:
        for start, width in zip(entry, (16, 8, 4)):
            assert start % width == 0
            used[start:start + width] += 1
    assert (used == 1).all()  # three blocks, full and without overlap
    for b in range(3):
        assert all(x % 128 == 0 for x in at[b * block])  # each row begins on a line
        for k, width in enumerate((16, 8, 4)):  # and is one stretch
            assert [e[k] for e in at[b * block:(b + 1) * block]] == [at[b * block][k] + width * j for j in range(block)]
    far = 4294967294
    assert max(last) < (far // block + 1) * size and min(last) >= far // block * size
