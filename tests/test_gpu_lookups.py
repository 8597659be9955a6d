"""wt_int lookups at the ends of the level bits: every position, the last directory
entry and the last word among them, and select's steps of four words."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def brute(s, i, j, c, c2):
    """rank, lex_count and range_count of each query (positions [i, j))."""
    below = np.array([(s[a:b] < v).sum() for a, b, v in zip(i, j, c)])
    upto = np.array([(s[a:b] <= v).sum() for a, b, v in zip(i, j, c2)])
    above = np.array([(s[a:b] > v).sum() for a, b, v in zip(i, j, c)])
    rank = np.array([(s[:a] == v).sum() for a, v in zip(i, c)])
    return rank, below, above, upto


@pytest.mark.parametrize("n,levels", [(1, 1), (1, 7), (63, 1), (64, 1), (64, 8), (65, 3), (512, 2), (513, 1), (1000, 9)])
def test_every_position(ctx, n, levels):
    rng = np.random.default_rng(n * 64 + levels)
    s = np.where(rng.random(n) < 0.8, 1, rng.integers(0, 1 << levels, n)).astype(np.uint64)
    wt = ctx.wtint_build(ctx.to_device(s), n, levels)
    at = np.arange(n, dtype=np.uint64)
    assert np.array_equal(wt.access(at), s)
    i = rng.integers(0, n + 1, 400).astype(np.uint64)
    j = rng.integers(0, n + 1, 400).astype(np.uint64)
    i, j = np.minimum(i, j), np.maximum(i, j)
    i[0], j[0], i[1], j[1] = 0, n, n, n
    c, c2 = (rng.integers(0, 1 << levels, 400).astype(np.uint64) for _ in range(2))
    c2[:100] = (1 << levels) - 1
    rank, below, above, upto = brute(s, i.astype(int), j.astype(int), c, c2)
    assert np.array_equal(wt.rank(i, c), rank)
    rk, sm, gr = wt.lex_count(i, j, c)
    assert np.array_equal(rk, rank) and np.array_equal(sm, below) and np.array_equal(gr, above)
    r, sm0 = wt.lex_smaller_count(i, c)
    assert np.array_equal(r, rank) and np.array_equal(sm0, [(s[:a] < v).sum() for a, v in zip(i.astype(int), c)])
    ok = (i < j) & (c <= c2)
    if ok.any():
        got = wt.range_count(i[ok], j[ok] - np.uint64(1), c[ok], c2[ok])
        assert np.array_equal(got, (upto - below)[ok])
    order = np.argsort(s, kind="stable")
    v = s[order]
    nth = (np.arange(n) - np.searchsorted(v, v) + 1).astype(np.uint64)
    assert np.array_equal(wt.select(nth, v), order)
    wt.free()
