"""Host parts of the library that need no GPU, compiled by themselves and run."""

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
PACKAGE = os.path.join(os.path.dirname(HERE), "higher_order_embedded_fem_amd")
CSRC = os.path.join(PACKAGE, "csrc")


def run(tmp_path, source):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(source)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


CHECK = """
#include <cstdio>
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\\n", __LINE__, #x); return 1; } } while (0)
"""


def test_resident_grids_are_admitted_in_order(tmp_path):
    """A launch that needs the whole device is not passed by later small ones, whether it waits or polls."""
    run(tmp_path, CHECK + """
#include <thread>
#include "cu_line.hpp"
using hoefem::CuLine;
int main() {
    CuLine L(16);
    const uint64_t a = L.enter();
    CHECK(L.take(a, 8, false));
    // one that waits in another thread
    const uint64_t wide = L.enter();
    std::thread t([&] { L.take(wide, 16, true); });
    const uint64_t small = L.enter();
    CHECK(!L.take(small, 4, false));  // 8 are free, but the wide one was first
    CHECK(!L.take_more(4));
    L.give(8);
    t.join();
    CHECK(!L.take(small, 4, false));  // all taken
    L.give(16);
    CHECK(L.take(small, 4, false));
    CHECK(L.take_more(12));
    CHECK(!L.take_more(1));
    L.give(16);
    // one that polls, and gives up
    const uint64_t b = L.enter();
    CHECK(L.take(b, 4, false));
    const uint64_t poll = L.enter();
    CHECK(!L.take(poll, 16, false));
    const uint64_t next = L.enter();
    CHECK(!L.take(next, 1, false));
    L.leave(poll);
    CHECK(L.take(next, 12, false));
    L.give(16);
    // small ones by turns from two threads while a wide one waits: it gets through
    auto churn = [&] {
        for (int i = 0; i < 20000; ++i) {
            const uint64_t p = L.enter();
            L.take(p, 6, true);
            L.give(6);
        }
    };
    std::thread c1(churn), c2(churn);
    for (int i = 0; i < 100; ++i) {
        const uint64_t p = L.enter();
        L.take(p, 16, true);
        L.give(16);
    }
    c1.join();
    c2.join();
    return 0;
}
""")


def test_admitted_grids_fit_every_xcd(tmp_path):
    """Every launch's work-groups go to the XCDs in turn from the first one: whatever is admitted together, no
    XCD gets more work-groups than it has CUs."""
    run(tmp_path, CHECK + """
#include <random>
#include <vector>
#include "cu_line.hpp"
using hoefem::CuLine;
int main() {
    std::mt19937 rng(1);
    for (int round = 0; round < 20000; ++round) {
        CuLine L(256);
        int xcd[8] = {};
        int sum = 0;
        for (int k = 0; k < 6; ++k) {
            const int wgs = round == 0 ? (k < 2 ? 82 : 90) : 1 + (int)(rng() % (round % 2 ? 256 : 100));
            const uint64_t p = L.enter();
            if (!L.take(p, CuLine::charge(wgs), false)) {
                L.leave(p);
                continue;
            }
            sum += wgs;
            for (int w = 0; w < wgs; ++w) ++xcd[w % 8];
        }
        CHECK(sum > 0 && sum <= 256);
        for (int x : xcd) CHECK(x <= 32);
    }
    CHECK(CuLine::charge(256) == 256 && CuLine::charge(1) == 8);
    return 0;
}
""")


def test_an_exception_in_a_worker_thread_reaches_the_caller(tmp_path):
    run(tmp_path, CHECK + """
#include <atomic>
#include <new>
#include <stdexcept>
#include "host_threads.hpp"
int main() {
    for (int n : {1, 2, 5, 8})
        for (int bad = -1; bad < n; ++bad) {  // the caller's own share is 0
            std::atomic<int> ran{0};
            bool caught = false;
            try {
                hoefem::run_on_threads(n, [&](int i) {
                    ++ran;
                    if (i == bad) throw std::bad_alloc();
                });
            } catch (const std::bad_alloc&) {
                caught = true;
            }
            CHECK(ran == n);
            CHECK(caught == (bad >= 0));
        }
    CHECK(hoefem::thread_count(0, 10) == 1 && hoefem::thread_count(1 << 30, 1) >= 1);
    return 0;
}
""")


def test_material_calls_of_short_lived_threads_leave_nothing_behind(tmp_path):
    """Threads one after the other use the same few pinned error words, and of many at a time a bounded number is kept
    (a thread may still be about to give its word back when join returns)."""
    stub = tmp_path / "libstub.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(stub), os.path.join(HERE, "hip_stub.c")], check=True)
    script = f"""
import ctypes as C, threading, time
S = C.CDLL({str(stub)!r}, mode=C.RTLD_GLOBAL)  # found before the HIP library's symbols
L = C.CDLL({os.path.join(PACKAGE, "libhoefem.so")!r})
L.hoefem_material_eval.argtypes = [C.c_double, C.c_double, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p]
buf = (C.c_double * 90)()
def call(times=1):
    for _ in range(times):
        assert L.hoefem_material_eval(1.0, 1.0, 1, C.addressof(buf), C.addressof(buf), None) == 0
before = S.stub_pinned_now()
for _ in range(50):
    t = threading.Thread(target=call)
    t.start()
    t.join()
    time.sleep(0.002)
assert S.stub_pinned_total() - before <= 16, S.stub_pinned_total()
ts = [threading.Thread(target=call, args=(200,)) for _ in range(40)]
for t in ts: t.start()
for t in ts: t.join()
time.sleep(0.2)
assert S.stub_pinned_now() - before <= 16, S.stub_pinned_now()
"""
    r = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
