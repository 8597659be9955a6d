"""Trees whose nodes get small before the last level: dense passes, then the small
nodes' remaining levels in one pass, large nodes of skewed inputs as a list of
segments.  Bits against the level-by-level split pipeline's definition (every
level = the stable sort by the top l bits), sigma against numpy."""
import numpy as np
import pytest

from test_gpu_levels_deep import closed_form

pytestmark = pytest.mark.gpu


def draw(rng, kind, n, L):
    top = (1 << L) - 1
    if kind == "uniform":
        return rng.integers(0, top, n, dtype=np.uint64, endpoint=True)
    if kind == "equal":
        return np.full(n, top // 3, np.uint64)
    if kind == "low":    # the top bits all zero: one node down to the last levels
        return rng.integers(0, min(top, 5), n, dtype=np.uint64, endpoint=True)
    # mixed: half of the keys in three values (nodes of thousands of keys down to
    # the last level), the others scattered
    s = rng.integers(0, top, n, dtype=np.uint64, endpoint=True)
    hot = rng.integers(0, top, 3, dtype=np.uint64, endpoint=True)
    pick = rng.random(n) < 0.5
    s[pick] = hot[rng.integers(0, 3, int(pick.sum()))]
    return s


@pytest.mark.parametrize("kind", ["uniform", "equal", "low", "mixed"])
@pytest.mark.parametrize("n,L,dt", [
    (1, 7, np.uint8), (65, 8, np.uint8), (2047, 16, np.uint16), (2048, 24, np.uint32), (2048, 64, np.uint64),
    (2049, 20, np.uint32), (3000, 33, np.uint64), (5003, 12, np.uint16), (40961, 18, np.uint32),
    (70001, 24, np.uint64), (300007, 32, np.uint32), (300007, 45, np.uint64), (1 << 18, 64, np.uint64)])
def test_small_nodes(ctx, kind, n, L, dt):
    rng = np.random.default_rng(n + L)
    s = draw(rng, kind, n, L).astype(dt)
    d = ctx.to_device(s)
    wt = ctx.wtint_build(d, n, L)
    try:
        assert wt.sigma == np.unique(s).size
        nw = (n * L + 63) // 64
        assert np.array_equal(wt.words()[:nw], closed_form(s, L)[:nw])
    finally:
        wt.free()
        d.free()
