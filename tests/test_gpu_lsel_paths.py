"""Learned select training: ten steps a launch against a launch for each half of a
step, the same knots to the last bit.  The second is taken for all vectors of a build
where one of them has too many samples for its knots (a vector of ones only)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def launches(ctx, build):
    ctx.kernel_timing_reset()
    ctx.kernel_timing(True)
    try:
        ls = build()
        return ls, ctx.kernel_time("lsel_train")[1], ctx.kernel_time("lsel_adam")[1]
    finally:
        ctx.kernel_timing(False)


@pytest.mark.parametrize("epochs", [1, 10, 11, 27])
def test_both_paths_give_the_same_knots(wsfm, ctx, epochs):
    rng = np.random.default_rng(epochs)
    nb = 1 << 22
    vecs = [rng.random(nb) < d for d in (0.03, 0.5, 0.2, 0.01)]
    vecs[2][nb // 3:nb // 2] = False
    vecs[3][nb // 2:] ^= rng.random(nb // 2) < 0.3
    vecs.append(np.ones(nb, bool))
    dv = [ctx.to_device(np.append(np.packbits(v, bitorder="little").view(np.uint64), np.uint64(0))) for v in vecs]
    par = wsfm.LselParams(16, 1 << 14, 64, epochs, 0.5, 512)
    one, steps, halves = launches(ctx, lambda: wsfm.LearnedSelect(ctx, dv[:4], [nb] * 4, par))
    assert steps == (epochs + 9) // 10 and halves == 0
    two, steps, halves = launches(ctx, lambda: wsfm.LearnedSelect(ctx, dv, [nb] * 5, par))
    assert steps == 0 and halves == epochs
    try:
        for b in range(4):
            (k1, l1, *m1), (k2, l2, *m2) = one.model(b), two.model(b)
            assert one.info(b)["trained"] == 1 and k1.size > 100
            assert np.array_equal(k1.view(np.uint64), k2.view(np.uint64)) and np.array_equal(l1, l2) and m1 == m2
            assert one.info(b) == two.info(b)
    finally:
        one.free()
        two.free()
        for d in dv:
            d.free()


@pytest.mark.parametrize("ones", [1, 20, 31])
def test_vectors_without_models(wsfm, ones):
    """Vectors of too few ones for a model, in a context that only enqueues: their tables'
    sources outlive the copies, and every query gets the plain answer."""
    rng = np.random.default_rng(ones)
    nb, nvec = 1 << 20, 200
    with wsfm.Context(0) as ctx:
        ctx.set_blocking(False)
        at = [np.sort(rng.choice(nb, ones, replace=False)) for _ in range(nvec)]
        dv = []
        for a in at:
            v = np.zeros(nb // 64 + 1, np.uint64)
            np.bitwise_or.at(v, a >> 6, np.uint64(1) << (a & 63).astype(np.uint64))
            dv.append(ctx.to_device(v))
        ls = wsfm.LearnedSelect(ctx, dv, [nb] * nvec)
        junk = [np.full(1 << 14, 0xFF, np.uint8) for _ in range(64)]  # (where freed sources lay)
        vec, j = np.repeat(np.arange(nvec, dtype=np.uint32), ones), np.tile(np.arange(1, ones + 1, dtype=np.uint64), nvec)
        for learned in (False, True):
            assert np.array_equal(ls.select(vec, j, learned=learned), np.concatenate(at))
        assert all(ls.info(b)["learned"] == 0 for b in range(nvec)) and len(junk) == 64
        ctx.sync()
        ls.free()
        for d in dv:
            d.free()
