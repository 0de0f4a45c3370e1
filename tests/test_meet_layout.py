"""Where the three arrays of a step's meetings begin in their allocation (stcdb_amd/csrc/stc_table.h): on 4 KB boundaries
whatever the capacity asked for, without overlap. The header alone is compiled, with the host's compiler."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stcdb_amd", "csrc")

PROGRAM = r"""
#include "stc_table.h"
#include <cstdio>
int main() {
    for (size_t n : {size_t(1), size_t(2), size_t(1023), size_t(1024), size_t(1025), size_t(98304), size_t(1234567), size_t(1577284626),
                     size_t(4294967294ull)}) {
        const MeetLayout l(n);
        printf("%zu %zu %zu %zu %zu\n", n, l.cap, l.keys, l.starts, l.bytes);
    }
    return 0;
}
"""


def test_arrays_begin_on_page_boundaries(tmp_path):
    src, exe = tmp_path / "layout.cpp", tmp_path / "layout"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True, timeout=120)
    rows = [tuple(map(int, line.split())) for line in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.splitlines()]
    assert len(rows) == 9
    for n, cap, keys, starts, size in rows:
        assert n <= cap < n + 1024
        assert keys % 4096 == 0 and starts % 4096 == 0
        assert keys >= 16 * cap and starts >= keys + 8 * cap and size >= starts + 4 * cap
