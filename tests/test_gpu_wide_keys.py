"""Trees of more than 24 levels over enough keys that the wide groups take 4096-key
tiles (above 32 levels the level loop moves the leaf and the key's place instead of
the key) and that the small nodes start below level 16: bits against the
level-by-level schedule's, sigma against numpy."""
import numpy as np
import pytest

from test_gpu_levels_deep import closed_form
from test_gpu_small_nodes import draw

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["uniform", "mixed", "low"])
@pytest.mark.parametrize("n,L,dt", [((1 << 21) + 4097, 40, np.uint64), ((1 << 21) + 1, 33, np.uint64), (6000011, 40, np.uint64),
                                    ((1 << 23) + 5, 26, np.uint32), ((1 << 24) + 77, 36, np.uint64)])
def test_large(ctx, kind, n, L, dt):
    s = draw(np.random.default_rng(n + L), kind, n, L).astype(dt)
    nw = (n * L + 63) // 64
    d, w = ctx.to_device(s), ctx.empty(nw)
    wt = ctx.wtint_build(d, n, L)
    try:
        got = wt.words()
        ctx.set_level_method(1)
        ctx.levels_build(d, n, L, w)
        assert np.array_equal(got, w.get())
        assert wt.sigma == np.unique(s).size
    finally:
        ctx.set_level_method(0)
        wt.free()
        d.free()
        w.free()


def test_split_schedule_itself(ctx):
    """The schedule that the larger trees are compared with, against the definition."""
    n, L = (1 << 18) + 9, 40
    s = draw(np.random.default_rng(1), "mixed", n, L)
    ctx.set_level_method(1)
    try:
        w, _ = ctx.levels(s, L)
    finally:
        ctx.set_level_method(0)
    assert np.array_equal(w, closed_form(s, L))


@pytest.mark.parametrize("n,values", [(2000003, 1000), (3000017, 1500), (6000011, 4000)])
@pytest.mark.parametrize("L,dt", [(24, np.uint32), (40, np.uint64)])
def test_many_large_nodes(ctx, n, values, L, dt):
    """Up to some thousands of values with 1500 to 2000 keys each: lists of large nodes on
    either side of the size that one launch makes the tables of."""
    rng = np.random.default_rng(n + L)
    s = rng.integers(0, (1 << L) - 1, values, dtype=np.uint64, endpoint=True)[rng.integers(0, values, n)].astype(dt)
    d, w, w1 = ctx.to_device(s), ctx.empty((n * L + 63) // 64), ctx.empty((n * L + 63) // 64)
    try:
        ctx.levels_build(d, n, L, w)
        ctx.set_level_method(1)
        ctx.levels_build(d, n, L, w1)
        assert np.array_equal(w.get(), w1.get())
        ctx.set_level_method(0)
        wt = ctx.wtint_build(d, n, L)
        assert wt.sigma == np.unique(s).size
        wt.free()
    finally:
        ctx.set_level_method(0)
        for x in (d, w, w1):
            x.free()
