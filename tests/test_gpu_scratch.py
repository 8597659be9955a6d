"""Scratch that a context keeps from call to call: it is given back on request, the
calls that use it work before and after, and it moves nothing that a recorded graph reads."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_levels_deep import closed_form

pytestmark = pytest.mark.gpu


def free_bytes(hip):
    f, t = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


def test_trim_gives_back(wsfm):
    n = 1 << 24
    t = wsfm.gen_dna(5, n)
    with wsfm.Context(0) as ctx:
        d, sa = ctx.to_device(t), ctx.empty(n, np.int64)
        run = lambda: wsfm._check(wsfm.lib().wtg_suffix_array_gpu(ctx.h, d.ptr, n, sa.ptr))  # noqa: E731
        run()
        first, held = sa.get(), free_bytes(wsfm.lib())
        assert np.bincount(first, minlength=n).max() == 1
        ctx.trim()
        assert free_bytes(wsfm.lib()) - held >= 40 * n
        ctx.trim()
        sa.zero()
        run()
        assert np.array_equal(sa.get(), first)
        d.free()
        sa.free()


def test_allocation_that_does_not_fit(wsfm):
    """An allocation larger than the device gives the scratch back, fails, and leaves the
    context usable; learned select, which allocates while it holds it, too."""
    n = 1 << 23
    t = wsfm.gen_dna(6, n)
    with wsfm.Context(0) as ctx:
        d, sa = ctx.to_device(t), ctx.empty(n, np.int64)
        run = lambda: wsfm._check(wsfm.lib().wtg_suffix_array_gpu(ctx.h, d.ptr, n, sa.ptr))  # noqa: E731
        run()
        first, held = sa.get(), free_bytes(wsfm.lib())
        with pytest.raises(wsfm.WtgError):
            ctx.empty(1 << 42, np.uint8)
        assert free_bytes(wsfm.lib()) - held >= 40 * n
        run()
        assert np.array_equal(sa.get(), first)
        bits = ctx.to_device(np.append(np.random.default_rng(2).integers(0, 1 << 63, 1 << 14).astype(np.uint64), np.uint64(0)))
        for _ in range(2):
            ls = wsfm.LearnedSelect(ctx, [bits], [1 << 20])
            assert ls.info(0)["nknots"] > 0
            ls.free()
            ctx.trim()
        for x in (d, sa, bits):
            x.free()


def test_recorded_graph_outlives_larger_scratch(wsfm):
    """A recorded tree build reads the workspace; a suffix array and a learned select
    built after it, both with more scratch, leave it where it is."""
    n, L = 70001, 20
    hip = wsfm.lib()
    with wsfm.Context(0) as ctx:
        stream = C.c_void_p(hip.wtg_ctx_stream(ctx.h))
        rng = np.random.default_rng(3)
        bits = ctx.to_device(np.append(rng.integers(0, 1 << 63, 1 << 14).astype(np.uint64), np.uint64(0)))
        wsfm.LearnedSelect(ctx, [bits], [1 << 20]).free()  # (its plain half uses the workspace)
        s = rng.integers(0, 1 << L, n).astype(np.uint32)
        d, w = ctx.to_device(s), ctx.empty((n * L + 63) // 64)
        ctx.levels_build(d, n, L, w)
        ctx.set_blocking(False)
        graph, run = C.c_void_p(), C.c_void_p()
        assert hip.hipStreamBeginCapture(stream, 1) == 0  # thread-local mode
        ctx.levels_build(d, n, L, w)
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
        assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
        ctx.set_blocking(True)
        want = closed_form(s, L)
        text = ctx.to_device(wsfm.gen_dna(5, 1 << 22))
        for _ in range(3):
            wsfm.suffix_array_gpu(ctx, text, 1 << 22).free()
            wsfm.LearnedSelect(ctx, [bits], [1 << 20]).free()
            w.zero()
            assert hip.hipGraphLaunch(run, stream) == 0
            ctx.sync()
            assert np.array_equal(w.get(), want)
        ctx.trim()
        w.zero()
        assert hip.hipGraphLaunch(run, stream) == 0
        ctx.sync()
        assert np.array_equal(w.get(), want)
        assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
        for x in (d, w, bits, text):
            x.free()
