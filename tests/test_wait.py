"""The short wait for a number that another thread (or the device) writes (stcdb_amd/csrc/stc_wait.h), on one core that it
shares with the thread that is to write it: the writer gets its turn while the wait lasts. Compiled with the host's
compiler."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stcdb_amd", "csrc")

PROGRAM = r"""
#include "stc_wait.h"
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <thread>
int main() {
    cpu_set_t set, one;
    if (sched_getaffinity(0, sizeof(set), &set)) return 1;
    int cpu = 0;
    while (!CPU_ISSET(cpu, &set)) cpu++;
    CPU_ZERO(&one);
    CPU_SET(cpu, &one);
    if (sched_setaffinity(0, sizeof(one), &one)) return 1;
    const int rounds = 200;
    std::atomic<int> asked{0}, written{0};
    std::thread writer([&] { /* has something to do all the time, as a thread that launches does */
        while (written < rounds) {
            if (asked > written) written++;
            else sched_yield();
        }
    });
    int in_time = 0;
    for (int r = 1; r <= rounds; r++) {
        asked = r;
        if (look_for([&] { return written >= r; }, std::chrono::microseconds(300))) in_time++;
        while (written < r) sched_yield();
    }
    writer.join();
    /* and a wait for nothing ends */
    const auto t0 = std::chrono::steady_clock::now();
    const bool none = look_for([] { return false; }, std::chrono::microseconds(300));
    const auto us = std::chrono::duration_cast<std::chrono::microseconds>(std::chrono::steady_clock::now() - t0).count();
    printf("%d %d %d\n", in_time, none ? 1 : 0, us >= 300 ? 1 : 0);
    return 0;
}
"""


def test_the_writer_gets_its_turn_on_the_same_core(tmp_path):
    src, exe = tmp_path / "wait.cpp", tmp_path / "wait"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I", CSRC, str(src), "-o", str(exe)], check=True, timeout=120)
    in_time, found, waited = map(int, subprocess.run([str(exe)], capture_output=True, text=True, timeout=120, check=True).stdout.split())
    assert found == 0 and waited == 1
    assert in_time > 100  # of 200: other processes share the core too
