"""Large host copies staged through pinned buffers: every byte arrives, and
nothing beside the destination is touched."""
import threading

import numpy as np
import pytest

from opsec_amd import lib, synth

pytestmark = pytest.mark.gpu
MB = 1 << 20


@pytest.fixture(scope="module")
def ctx():
    """A context whose slots are made: its first large copy pays for them."""
    with lib.Context(0) as c:
        p = c.dev_alloc(128 * MB)
        c.h2d(p, np.zeros(128 * MB, dtype=np.uint8))
        c.dev_free(p)
        yield c


# under, at and over the least staged sizes (8 MB to the host, 32 MB to the device);
# full 4 MB chunks with a last partial one, more of them than threads
@pytest.mark.parametrize("n", [1, 8 * MB - 1, 8 * MB, 8 * MB + 1, 32 * MB - 1, 32 * MB, 32 * MB + 1, 70 * MB + 5])
def test_round_trip_bytes(ctx, n):
    src = np.random.default_rng(n).integers(0, 256, n, dtype=np.uint8)
    p = ctx.dev_alloc(n)
    try:
        ctx.h2d(p, src)
        frame = np.full(n + 130, 7, dtype=np.uint8)   # an odd host address
        ctx.d2h(frame[65:65 + n], p)
        assert np.array_equal(frame[65:65 + n], src)
        assert np.all(frame[:65] == 7) and np.all(frame[65 + n:] == 7)
        ctx.h2d(p, src[::-1].copy())                   # the buffers again, other bytes
        back = np.empty(n, dtype=np.uint8)
        ctx.d2h(back, p)
        assert np.array_equal(back, src[::-1])
    finally:
        ctx.dev_free(p)


def test_two_threads(ctx):
    """Copies of two threads at once: one has the buffers, the other goes by the runtime."""
    n = 40 * MB + 1
    rng = np.random.default_rng(5)
    srcs = [rng.integers(0, 256, n, dtype=np.uint8) for _ in range(2)]
    outs = [np.zeros(n, dtype=np.uint8) for _ in range(2)]
    ptrs = [ctx.dev_alloc(n) for _ in range(2)]

    def run(i):
        ctx.h2d(ptrs[i], srcs[i])
        ctx.d2h(outs[i], ptrs[i])

    try:
        th = [threading.Thread(target=run, args=(i,)) for i in range(2)]
        for t in th:
            t.start()
        for t in th:
            t.join()
        assert np.array_equal(outs[0], srcs[0]) and np.array_equal(outs[1], srcs[1])
    finally:
        for p in ptrs:
            ctx.dev_free(p)


def test_first_copies_of_a_context():
    """The runtime's copies, the one that makes the slots, and the staged ones after it."""
    n = 40 * MB + 3
    rng = np.random.default_rng(6)
    with lib.Context(0) as c:
        p = c.dev_alloc(n)
        for _ in range(5):
            src = rng.integers(0, 256, n, dtype=np.uint8)
            c.h2d(p, src)
            back = np.empty(9 * MB, dtype=np.uint8)
            c.d2h(back, p)
            assert np.array_equal(back, src[:9 * MB])
        c.dev_free(p)


def test_refused_allocation_leaves_the_context_usable():
    """More memory than there is: the call fails, and the launches of the next ones are not
    blamed for it, through every path that allocates."""
    cells = synth.box_cells(2, 0.0, 20.0)
    sv = lib.survey_box(2, 0.0, 20.0, L=1e9)
    with lib.Context(0) as c:
        c.model_test(0, 1.0, 0.1)
        c.cells_upload(cells, sv)
        q = c.quad(lib.OPSEC_QUAD_GAUSS, nodes=4, near=1)
        with pytest.raises(lib.OpsecError):
            c.dev_alloc(1 << 50)
        c.pair_tables([0], q)
        S = c.assemble(0, len(cells))
        with pytest.raises(lib.OpsecError):   # its buffer on the device; the host's S is never read
            c.check(c.lib.opsec_project_dense(c.h, 1 << 20, S.ctypes.data, 2, S.ctypes.data, 0, S.ctypes.data))
        got = c.project_dense(S, np.eye(8), lib.OPSEC_PREC_FP64)
        assert np.array_equal(got, [S[i, j] for j in range(8) for i in range(j + 1)])
