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


@pytest.fixture(scope="module")
def large(ctx):
    """2^26 level bits: batches of 2^18 queries on it are put in order."""
    n, levels = (1 << 26) // 9 + 1, 9
    s = np.random.default_rng(5).integers(0, 1 << levels, n)
    s[::3] = 77
    wt = ctx.wtint_build(ctx.to_device(s.astype(np.uint32)), n, levels)
    yield wt
    wt.free()


@pytest.mark.parametrize("nq", [1 << 18, (1 << 18) + 2049, (1 << 20) + 3])
@pytest.mark.parametrize("keys", ["any", "one", "few", "refused"])
def test_ordered_batch(ctx, large, nq, keys):
    """A batch in order gives what the same queries give in small batches, as they came."""
    wt, rng = large, np.random.default_rng(nq)
    n, top = wt.n, 1 << wt.L
    i, j = (rng.integers(0, n + 3, nq).astype(np.uint64) for _ in range(2))
    lo, hi = (rng.integers(0, top + 2, nq).astype(np.uint64) for _ in range(2))
    k = rng.integers(0, 3000, nq).astype(np.uint64)
    if keys == "one":
        i[:], lo[:] = n // 2, 77
    elif keys == "few":
        i, lo = i % np.uint64(3), lo % np.uint64(3)
    elif keys == "refused":
        i[::2], lo[::2], hi[::2] = n + 1, 1 << 62, np.uint64(2**64 - 1)
    calls = [(wt.rank, (i, lo)), (wt.access, (i,)), (wt.inverse_select, (i,)), (wt.lex_count, (i, j, lo)),
             (wt.lex_smaller_count, (i, lo)), (wt.range_count, (i, j, lo, hi)), (wt.select, (k, lo))]
    step = 100000
    for f, a in calls:
        got = f(*a)
        parts = [f(*(x[at:at + step] for x in a)) for at in range(0, nq, step)]
        if isinstance(got, list):
            want = [np.concatenate([p[c] for p in parts]) for c in range(len(got))]
            assert all(np.array_equal(g, w) for g, w in zip(got, want)), f.__name__
        else:
            assert np.array_equal(got, np.concatenate(parts)), f.__name__


def test_ordered_answers_over_their_queries(ctx, large):
    """Answers written over a column of the batch itself."""
    from wavelet_suffix_fm_index_amd import _check, lib
    wt, rng, nq = large, np.random.default_rng(1), 1 << 18
    lb, rb = np.sort(rng.integers(0, wt.n, (2, nq)), axis=0).astype(np.uint64)
    lo, hi = np.sort(rng.integers(0, 1 << wt.L, (2, nq)), axis=0).astype(np.uint64)
    want = wt.range_count(lb, rb, lo, hi)
    ranks = wt.rank(lb, lo)
    for over in range(4):
        d = [ctx.to_device(x) for x in (lb, rb, lo, hi)]
        _check(lib().wtg_wtint_range_count_batch(ctx.h, wt.h, *[x.ptr for x in d], nq, d[over].ptr))
        assert np.array_equal(d[over].get(), want)
        for x in d:
            x.free()
    d = [ctx.to_device(x) for x in (lb, lo)]
    _check(lib().wtg_wtint_rank_batch(ctx.h, wt.h, d[0].ptr, d[1].ptr, nq, d[1].ptr))
    assert np.array_equal(d[1].get(), ranks)
    for x in d:
        x.free()


@pytest.mark.parametrize("m", [12, 13, 32])
def test_ordered_patterns(ctx, m):
    """A batch of patterns in order gives the counts of the same patterns in small
    batches, as they came (2^26 code bits, 16 symbols, some patterns of absent ones)."""
    rng = np.random.default_rng(m)
    n = (1 << 24) + 1
    wt = ctx.huff_build(ctx.to_device((rng.integers(0, 16, n) * 3).astype(np.uint8)))
    try:
        for nq in (1 << 19, (1 << 20) + 5):
            pats = (rng.integers(0, 16, (nq, m)) * 3).astype(np.uint8)
            pats[:, :m - 5] = pats[rng.integers(0, 50, nq), :m - 5]  # some counts stay above 0
            pats[::7, -1] = 1
            pats[5::7, 0] = 255
            got = wt.fm_count(pats)
            step = 1 << 18
            assert np.array_equal(got, np.concatenate([wt.fm_count(pats[at:at + step]) for at in range(0, nq, step)]))
    finally:
        wt.free()


@pytest.fixture(scope="module")
def wide(ctx):
    """2^26 level bits in 16 levels: symbol batches of 2^18 queries are put in order."""
    n = (1 << 22) + 5
    s = np.random.default_rng(6).integers(0, 1 << 16, n)
    s[::3] = 777
    wt = ctx.wtint_build(ctx.to_device(s.astype(np.uint16)), n, 16)
    yield wt
    wt.free()


def in_runs(rng, x, runs, down):
    """x rearranged as `runs` sorted stretches of one length, up or down."""
    x = np.array_split(rng.permutation(x), runs)
    return np.concatenate([np.sort(p)[::-1] if down else np.sort(p) for p in x])


@pytest.mark.parametrize("nq", [1 << 18, (1 << 20) + 5])
@pytest.mark.parametrize("runs,down", [(1, False), (1, True), (15, False), (16, True), (17, False), (40, True)])
def test_batch_in_order(ctx, wide, nq, runs, down):
    """Batches that come in order, up or down, in few runs or in more than count as order,
    give what the same queries give in small batches, as they came."""
    wt, rng = wide, np.random.default_rng(nq + runs)
    n, top = wt.n, 1 << wt.L
    i, j = (in_runs(rng, rng.integers(0, n, nq).astype(np.uint64), runs, down) for _ in range(2))
    lo, hi = (in_runs(rng, rng.integers(0, top, nq).astype(np.uint64), runs, down) for _ in range(2))
    k = rng.integers(1, 3000, nq).astype(np.uint64)
    calls = [(wt.rank, (i, lo)), (wt.access, (i,)), (wt.inverse_select, (i,)), (wt.lex_count, (np.minimum(i, j), np.maximum(i, j), lo)),
             (wt.lex_smaller_count, (i, lo)), (wt.range_count, (np.minimum(i, j), np.maximum(i, j), lo, rng.permutation(hi))),
             (wt.select, (k, lo))]
    step = 100000
    for f, a in calls:
        got = f(*a)
        parts = [f(*(x[at:at + step] for x in a)) for at in range(0, nq, step)]
        if isinstance(got, list):
            want = [np.concatenate([p[c] for p in parts]) for c in range(len(got))]
            assert all(np.array_equal(g, w) for g, w in zip(got, want)), f.__name__
        else:
            assert np.array_equal(got, np.concatenate(parts)), f.__name__


@pytest.mark.parametrize("m", [12, 19, 32])
def test_patterns_in_order(ctx, m):
    """Patterns in the order of their last eight bytes (last byte first), up and down, and
    one pattern over and over: counts as in small batches."""
    rng = np.random.default_rng(m)
    n = (1 << 24) + 1
    wt = ctx.huff_build(ctx.to_device((rng.integers(0, 16, n) * 3).astype(np.uint8)))
    try:
        nq = (1 << 20) + 5
        pats = (rng.integers(0, 16, (nq, m)) * 3).astype(np.uint8)
        pats[:, :m - 5] = pats[rng.integers(0, 50, nq), :m - 5]
        key = np.ascontiguousarray(pats[:, m - 8:]).view("<u8").reshape(-1)
        up = pats[np.argsort(key, kind="stable")]
        for p in (up, up[::-1], np.repeat(pats[:1], nq, 0), np.concatenate([up[::7]] * 7)[:nq]):
            got, step = wt.fm_count(p), 1 << 18
            assert np.array_equal(got, np.concatenate([wt.fm_count(p[at:at + step]) for at in range(0, p.shape[0], step)]))
    finally:
        wt.free()


def test_captured_batches(wsfm, ctx, wide):
    """Large batches recorded as a graph (answered as they come, with no block shared with
    other work), replayed over other queries in the same place."""
    import ctypes as C
    hip, wt, nq = wsfm.lib(), wide, 1 << 18
    stream = C.c_void_p(hip.wtg_ctx_stream(ctx.h))
    rng = np.random.default_rng(9)
    i, c, out, inv = (ctx.empty(nq) for _ in range(4))
    i.zero()
    c.zero()
    graph, run = C.c_void_p(), C.c_void_p()
    ctx.set_blocking(False)
    try:
        assert hip.hipStreamBeginCapture(stream, 1) == 0  # thread-local mode
        wsfm._check(hip.wtg_wtint_rank_batch(ctx.h, wt.h, i.ptr, c.ptr, nq, out.ptr))
        wsfm._check(hip.wtg_wtint_access_batch(ctx.h, wt.h, i.ptr, nq, inv.ptr))
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    finally:
        ctx.set_blocking(True)
    assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    for _ in range(3):
        qi, qc = rng.integers(0, wt.n, nq).astype(np.uint64), rng.integers(0, 1 << wt.L, nq).astype(np.uint64)
        for d, q in ((i, qi), (c, qc)):
            wsfm._check(hip.wtg_memcpy_h2d(ctx.h, d.ptr, C.c_void_p(q.ctypes.data), q.nbytes))
        assert hip.hipGraphLaunch(run, stream) == 0
        ctx.sync()
        assert np.array_equal(out.get(), wt.rank(qi, qc)) and np.array_equal(inv.get(), wt.access(qi))
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    for x in (i, c, out, inv):
        x.free()


@pytest.mark.parametrize("levels", [2, 4, 8, 11])
def test_large_batch_on_few_levels(ctx, levels):
    """2^26 level bits in few levels, batches on either side of 2^18 queries: large ones
    walk a lookup at a time; answers against the small batches'."""
    rng = np.random.default_rng(levels)
    n, top = (1 << 26) // levels + 3, 1 << levels
    wt = ctx.wtint_build(ctx.to_device(np.minimum(rng.geometric(0.2, n) - 1, top - 1).astype(np.uint16)), n, levels)
    try:
        for nq in ((1 << 18) - 1, 1 << 18, (1 << 20) + 1):
            i, j = np.sort(rng.integers(0, n, (2, nq)), axis=0).astype(np.uint64)
            lo, hi = np.sort(rng.integers(0, top + 1, (2, nq)), axis=0).astype(np.uint64)
            step = 100000
            for f, a in ((wt.rank, (i, lo)), (wt.access, (i,)), (wt.lex_count, (i, j, lo)), (wt.lex_smaller_count, (i, lo)),
                         (wt.range_count, (i, j, lo, hi)), (wt.select, (np.uint64(1) + i % np.uint64(5000), lo))):
                got = f(*a)
                parts = [f(*(x[at:at + step] for x in a)) for at in range(0, nq, step)]
                got, parts = ([got], [[p] for p in parts]) if not isinstance(got, list) else (got, parts)
                assert all(np.array_equal(g, np.concatenate([p[c] for p in parts])) for c, g in enumerate(got)), f.__name__
    finally:
        wt.free()


@pytest.mark.parametrize("nq", [1 << 18, (1 << 19) + 2049])
@pytest.mark.parametrize("keys", ["any", "one", "few", "refused"])
def test_ordered_batch_on_many_levels(ctx, wide, nq, keys):
    test_ordered_batch(ctx, wide, nq, keys)


def test_ordered_answers_over_their_queries_on_many_levels(ctx, wide):
    test_ordered_answers_over_their_queries(ctx, wide)
