"""Trees whose nodes get small before the last level, in contexts that only enqueue:
the call does not wait for the stream, and the rounds over large nodes, launched
without knowing how many there are, give the same bits; eagerly and as a graph."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_levels_deep import closed_form
from test_gpu_small_nodes import draw

pytestmark = pytest.mark.gpu
NOT_READY = 600  # hipErrorNotReady


@pytest.fixture
def queueing(wsfm):
    c = wsfm.Context(0)
    c.set_blocking(False)
    yield c
    c.sync()
    c.close()


@pytest.mark.parametrize("kind", ["uniform", "mixed"])
@pytest.mark.parametrize("n,L,dt", [(3000, 20, np.uint32), (300007, 24, np.uint32), (300007, 45, np.uint64)])
def test_build_only_enqueues(wsfm, queueing, kind, n, L, dt):
    ctx, hip = queueing, wsfm.lib()  # (its HIP runtime's names are found through it)
    stream = C.c_void_p(hip.wtg_ctx_stream(ctx.h))
    s = draw(np.random.default_rng(n + L), kind, n, L).astype(dt)
    d, w = ctx.to_device(s), ctx.empty((n * L + 63) // 64)
    big = ctx.to_device(np.random.default_rng(1).integers(0, 1 << 16, 1 << 24).astype(np.uint32))
    bw = ctx.empty((big.size * 16) // 64)
    ctx.levels_build(d, n, L, w)  # (the workspace grows here)
    ctx.levels_build(big, big.size, 16, bw)
    ctx.sync()
    w.zero()
    for _ in range(60):  # some 20 ms of work before it
        ctx.levels_build(big, big.size, 16, bw)
    before = C.c_void_p()
    assert hip.hipEventCreate(C.byref(before)) == 0 and hip.hipEventRecord(before, stream) == 0
    ctx.levels_build(d, n, L, w)
    waiting = hip.hipEventQuery(before)
    ctx.sync()
    assert hip.hipEventQuery(before) == 0 and hip.hipEventDestroy(before) == 0
    assert np.array_equal(w.get(), closed_form(s, L))
    assert waiting == NOT_READY
    for x in (d, w, big, bw):
        x.free()


@pytest.mark.parametrize("kind", ["uniform", "equal", "low", "mixed"])
@pytest.mark.parametrize("n,L,dt", [(2049, 20, np.uint32), (70001, 24, np.uint64), (300007, 32, np.uint32), (100003, 64, np.uint64)])
def test_rounds_launched_unasked(queueing, kind, n, L, dt):
    ctx = queueing
    s = draw(np.random.default_rng(n + L), kind, n, L).astype(dt)
    d, w = ctx.to_device(s), ctx.empty((n * L + 63) // 64)
    ctx.levels_build(d, n, L, w)
    wt = ctx.wtint_build(d, n, L)
    ctx.sync()
    want = closed_form(s, L)
    assert np.array_equal(w.get(), want)
    assert wt.sigma == np.unique(s).size and np.array_equal(wt.words(), want)
    wt.free()
    d.free()
    w.free()


@pytest.mark.parametrize("kind", ["uniform", "mixed"])
@pytest.mark.parametrize("n,L,dt", [(70001, 24, np.uint32), (100003, 40, np.uint64)])
def test_captured_build(wsfm, queueing, kind, n, L, dt):
    """A build recorded as a graph, replayed over new keys in the same place."""
    ctx, hip = queueing, wsfm.lib()
    stream = C.c_void_p(hip.wtg_ctx_stream(ctx.h))
    rng = np.random.default_rng(n + L)
    d, w = ctx.empty(n, dt), ctx.empty((n * L + 63) // 64)
    d.zero()
    ctx.levels_build(d, n, L, w)  # (the workspace grows here)
    ctx.sync()
    graph, run = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 1) == 0  # thread-local mode
    ctx.levels_build(d, n, L, w)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    for _ in range(4):
        s = draw(rng, kind, n, L).astype(dt)
        wsfm._check(hip.wtg_memcpy_h2d(ctx.h, d.ptr, C.c_void_p(s.ctypes.data), s.nbytes))
        w.zero()
        assert hip.hipGraphLaunch(run, stream) == 0
        ctx.sync()
        assert np.array_equal(w.get(), closed_form(s, L))
        ctx.levels_build(d, n, L, w)
        ctx.sync()
        assert np.array_equal(w.get(), closed_form(s, L))
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    d.free()
    w.free()
