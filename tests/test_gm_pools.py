"""Region pools of the adaptive cubature: how many, how large, and what is tried
when the memory is not there.  CPU only: the host rule through its diagnostic."""
import ctypes as C

import pytest

from opsec_amd import lib

CUS, CAP = 256, 50000000
WHOLE = CAP // 149 + 2
REGION, POOL, GB = 144, 1024, 1 << 30


def pools(rerun, n, maxeval=CAP, free=280 * GB, held=0, cap=0, failures=0):
    out = (C.c_int * 3)()
    rc = lib.load().opsec_diag_gm_pools(rerun, n, CUS, maxeval, free, held, cap, failures, out)
    return tuple(out) if rc == 0 else rc


def test_first_pools_whole_only_within_bounds():
    most = 2 * GB // (WHOLE * REGION)
    assert most < CUS
    assert pools(0, 1) == (WHOLE, 1, 1)
    assert pools(0, most) == (WHOLE, most, 1)
    assert pools(0, most + 1) == (POOL, most + 1, 0)
    assert pools(0, CUS, maxeval=10000) == (69, CUS, 1)        # small pools: one per CU
    assert pools(0, CUS + 1, maxeval=10000) == (POOL, CUS + 1, 0)
    assert pools(0, 10 ** 6) == (POOL, 8 * CUS, 0)
    need = most * WHOLE * REGION
    assert pools(0, most, free=4 * need)[2] == 1
    assert pools(0, most, free=4 * need - 4) == (POOL, most, 0)
    # the sweep's own pools of an earlier chunk can be used again
    assert pools(0, 2 * most, free=0, held=2 * need)[2] == 1
    # two sweeps that see the same free memory take at most half of it together
    for free in (GB, 3 * GB, 20 * GB, 48 * GB, 280 * GB):
        for n in (1, 7, 40, CUS, 5000):
            r, slots, whole = pools(0, n, free=free)
            assert not whole or 2 * r * slots * REGION <= free // 2
            assert r * slots * REGION <= 2 * GB


def test_rerun_takes_half_the_free_memory_and_the_cap():
    assert pools(1, 5) == (WHOLE, 5, 1)
    assert pools(1, 5000) == (WHOLE, 8 * CUS, 1)
    assert pools(1, 5000, free=4 * GB)[1] == 2 * GB // (WHOLE * REGION)
    assert pools(1, 5000, free=0)[1] == GB // (WHOLE * REGION)
    assert pools(1, 5000, cap=3 * CUS) == (WHOLE, 3 * CUS, 1)
    assert pools(1, 3, maxeval=2 ** 31 - 1, free=0) == (1 << 22, 1, 1)


@pytest.mark.parametrize("maxeval,regions", [(0, 1 << 20), (2 ** 31 - 1, 1 << 22), (CAP, WHOLE)])
def test_running_out_of_a_whole_pool_is_final(maxeval, regions):
    """No second sweep with the same pools: `whole` says that the first one decides."""
    assert pools(0, 3, maxeval=maxeval) == (regions, 3, 1) == pools(1, 3, maxeval=maxeval)
    assert pools(0, CUS + 1, maxeval=maxeval)[2] == 0


def test_smaller_pools_when_the_memory_is_not_there():
    assert pools(0, 20)[2] == 1 and pools(0, 20, failures=1) == (POOL, 20, 0)
    seen = [pools(0, 200, failures=k) for k in range(1, 9)]
    assert seen == [(POOL, s, 0) for s in (100, 50, 25, 13, 7, 4, 2, 1)]
    assert pools(0, 200, failures=9) == -2 and pools(0, 20, failures=7) == -2
    assert pools(1, 3, failures=1) == (WHOLE, 2, 1) and pools(1, 3, failures=2) == (WHOLE, 1, 1)
    assert pools(1, 3, failures=3) == -2
