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
// a runtime whose call number `fail` (a slot's allocation, its event, the next slot's) fails and
// leaves an error
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
    const int want = std::atoi(v[2]);
    opsec::StageSlots<Api> s;
    const int got = s.make(want);
    std::printf("%d %d %d %d ", got, Api::error, Api::live_mem, Api::live_ev);
    const int again = s.make(s.N), calls = Api::calls;   // the failed call has passed
    const int fewer = s.make(3);
    std::printf("%d %d %d %d %d ", again, Api::error, fewer, calls == Api::calls, Api::live_mem);
    s.release();
    std::printf("%d %d\n", Api::live_mem, Api::live_ev);
}
"""


@pytest.fixture(scope="module")
def prog(tmp_path_factory):
    d = tmp_path_factory.mktemp("stage")
    (d / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "opsec_amd", "csrc"), "-o",
                    str(d / "t"), str(d / "t.cpp")], check=True)
    return str(d / "t")


@pytest.mark.parametrize("want", [1, 5, 8])
@pytest.mark.parametrize("fail", range(-1, 17))
def test_failed_slots_leave_no_error(prog, fail, want):
    """Whichever call fails (each slot's allocation, then its event; -1: none), the slots before
    it are kept, nothing else is held, no error is left behind, and the next call goes on."""
    out = [int(x) for x in subprocess.run([prog, str(fail), str(want)], capture_output=True, text=True,
                                          check=True).stdout.split()]
    got = want if fail < 0 else min(want, fail // 2)
    assert out[:4] == [got, 0, got, got]
    again = 8 if fail < 0 or got < want or fail >= 16 else fail // 2   # it fails on the second call
    assert out[4:] == [again, 0, 3, int(again >= 3), max(3, again), 0, 0]   # then three are there
