"""Set-up of the staging slots of large host copies, its failures included: compiled
for the CPU against a stand-in for the runtime's calls."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "stage.h"
// a runtime whose call number `fail` (allocation, then the events) fails and leaves an error
struct Api {
    typedef int event_t;
    static int calls, fail, error, live_mem, live_ev;
    static bool call() {
        if (calls++ != fail) return true;
        error = 1;
        return false;
    }
    static bool host_alloc(void** p, size_t n) {
        if (!call()) return false;
        live_mem++;
        *p = std::malloc(n);
        return true;
    }
    static void host_free(void* p) { live_mem--; std::free(p); }
    static bool event_create(int* e) {
        if (!call()) return false;
        *e = ++live_ev;
        return true;
    }
    static void event_destroy(int) { live_ev--; }
    static void clear_error() { error = 0; }
};
int Api::calls, Api::fail, Api::error, Api::live_mem, Api::live_ev;

int main(int, char** v) {
    Api::fail = std::atoi(v[1]);
    opsec::StageSlots<Api> s;
    const bool first = s.make();
    std::printf("%d %d %d %d ", first, Api::error, Api::live_mem, Api::live_ev);
    const bool again = s.make();   // the failed call has passed
    const int calls = Api::calls, third = s.make();
    const int disjoint = s.slot(s.N - 1) + s.BYTES <= s.base + s.N * s.BYTES && s.slot(1) >= s.slot(0) + s.BYTES;
    std::printf("%d %d %d %d", again, Api::error, third && calls == Api::calls, disjoint);
    s.release();
    std::printf(" %d %d\n", Api::live_mem, Api::live_ev);
}
"""


@pytest.fixture(scope="module")
def prog(tmp_path_factory):
    d = tmp_path_factory.mktemp("stage")
    (d / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "opsec_amd", "csrc"), "-o",
                    str(d / "t"), str(d / "t.cpp")], check=True)
    return str(d / "t")


@pytest.mark.parametrize("fail", range(-1, 9))
def test_no_slots_and_no_error_left(prog, fail):
    """Whichever call fails (-1: none), there are all slots or none, nothing is held, no error
    is left behind, and the next call makes the slots."""
    out = subprocess.run([prog, str(fail)], capture_output=True, text=True, check=True).stdout.split()
    ok = fail < 0
    assert out[:4] == (["1", "0", "1", "8"] if ok else ["0", "0", "0", "0"])
    assert out[4:] == ["1", "0", "1", "1", "0", "0"]
