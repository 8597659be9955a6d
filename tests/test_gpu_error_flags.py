"""Device-side error flags: every call that meets an error reports it, however many
waves found it, one after the other and between calls that are right, in one context
and in two, waited for by the call or later."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def build(ctx, s, L):
    d, w = ctx.to_device(s), ctx.empty((s.size * L + 63) // 64)
    try:
        ctx.levels_build(d, s.size, L, w)
        ctx.sync()
        return w.get()
    finally:
        d.free()
        w.free()


@pytest.mark.parametrize("n,L,dt", [(5003, 5, np.uint8), (100003, 5, np.uint8), (1 << 21, 12, np.uint16), (70001, 20, np.uint32),
                                    (70001, 40, np.uint64)])
@pytest.mark.parametrize("blocking", [True, False])
def test_every_error_is_reported(wsfm, n, L, dt, blocking):
    rng = np.random.default_rng(n + L)
    good = rng.integers(0, 1 << L, n, dtype=np.uint64).astype(dt)
    every, one = good | dt(1 << L), good.copy()
    one[n // 2] |= dt(1 << L)
    with wsfm.Context(0) as a, wsfm.Context(0) as b:
        a.set_blocking(blocking)
        b.set_blocking(blocking)
        want = build(a, good, L)
        for bad in (every, one, every, every, one, one):
            with pytest.raises(wsfm.WtgError, match="levels"):
                build(a, bad, L)
            assert np.array_equal(build(b, good, L), want)
            a.sync()
            b.sync()
        with pytest.raises(wsfm.WtgError):
            build(b, every, L)
        assert np.array_equal(build(a, good, L), want)
        assert np.array_equal(build(b, good, L), want)


def test_flags_of_two_kinds(wsfm, ctx):
    """A suffix array that is none, between symbols out of range."""
    n = 1 << 20
    t = ctx.to_device(np.full(n, 65, np.uint8))
    bad = ctx.to_device(np.full(n, 1 << 40, np.int64))
    s = np.full(20000, 255, np.uint8)
    for _ in range(3):
        with pytest.raises(wsfm.WtgError, match="suffix array"):
            wsfm.bwt_from_sa_gpu(ctx, t, bad, n)
        with pytest.raises(wsfm.WtgError, match="levels"):
            build(ctx, s, 3)
    ctx.sync()
    t.free()
    bad.free()
