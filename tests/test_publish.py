"""The published state that query batches read while steps go on (stcdb_amd/csrc/stc_serve.h): whatever a step frees or
overwrites is no longer named by any lease. The header alone is compiled here, with the host's compiler."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stcdb_amd", "csrc")

PROGRAM = r"""
#include "stc_serve.h"
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <thread>
struct Array { std::atomic<int> freed{0}; };
struct State { Array *rec = nullptr; Array *meet = nullptr; };
using Pub = Published<State>;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); exit(1); } } while (0)
static void nap(int ms) { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); }

/* growth: the new array is named before the old one goes, which waits for the leases on it and for no later one */
static void growth() {
    Pub p;
    Array a, b;
    Pub::Lease old, later;
    CHECK(!p.take(&old));
    p.publish(State{&a, nullptr}, 0, 0, true);
    CHECK(p.take(&old) && old.state.rec == &a);
    std::atomic<int> gone{0};
    std::thread step([&] {
        p.replace([&](State &s) { s.rec = &b; }, [&] { gone = 1; });
        gone = 2;
    });
    nap(30);
    CHECK(gone == 0);                                     /* the lease still reads a */
    CHECK(p.take(&later) && later.state.rec == &b);       /* a batch admitted after the growth sees the new array */
    p.give_back(old);
    step.join();                                          /* although `later` is open */
    CHECK(gone == 2);
    p.give_back(later);
    p.wait_all();
}

/* overwriting: a state that still names the array or the records is withdrawn until the next publish */
static void overwriting() {
    Pub p;
    Array a, b;
    Pub::Lease l;
    p.publish(State{nullptr, &a}, 0, 4, true);
    p.clear(1, false, 4);
    CHECK(p.take(&l));                                    /* array 1 is not the published one */
    std::atomic<int> done{0};
    std::thread step([&] { p.clear(0, false, 4); done = 1; });
    nap(30);
    CHECK(done == 0);
    Pub::Lease x;
    CHECK(!p.take(&x));                                   /* and none comes in meanwhile, nor after it */
    p.give_back(l);
    step.join();
    CHECK(!p.take(&x));
    p.publish(State{nullptr, &b}, 1, 4, true);
    CHECK(p.take(&x) && x.state.meet == &b);
    p.give_back(x);
    p.clear(0, true, 4);
    CHECK(p.take(&x));
    p.give_back(x);
    p.clear(0, true, 5);                                  /* records of an epoch before */
    CHECK(!p.take(&x));
    p.publish(State{}, 0, 0, false);
    CHECK(!p.take(&x));
}

/* batches without a pause against steps that grow, overwrite and publish: no batch meets an array that is gone */
static void traffic() {
    Pub p;
    Array *meet[2] = {new Array, new Array}, *rec = new Array;
    std::atomic<int> stop{0}, seen{0};
    p.publish(State{rec, meet[0]}, 0, 0, true);
    auto query = [&] {
        while (!stop) {
            Pub::Lease l;
            if (!p.take(&l)) continue;
            for (int k = 0; k < 50; k++) CHECK(!l.state.rec->freed && !l.state.meet->freed);
            seen++;
            p.give_back(l);
        }
    };
    std::thread q1(query), q2(query);
    int cur = 0;
    for (int t = 0; t < 3000 || seen < 2000; t++) {
        const int nx = cur ^ 1;
        Array *grown = new Array, *was = rec;
        p.replace([&](State &s) { s.rec = grown; }, [&] { was->freed = 1; });
        rec = grown;
        p.clear(nx, false, 0);
        meet[nx]->freed = 1;
        meet[nx] = new Array;
        cur = nx;
        p.publish(State{rec, meet[cur]}, cur, 0, true);
    }
    stop = 1;
    q1.join();
    q2.join();
}

int main() {
    growth();
    overwriting();
    traffic();
    printf("ok\n");
    return 0;
}
"""


def test_nothing_a_lease_names_is_freed(tmp_path):
    src, exe = tmp_path / "publish.cpp", tmp_path / "publish"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I", CSRC, str(src), "-o", str(exe)], check=True,
                   timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
