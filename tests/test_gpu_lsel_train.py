"""Several training steps of the learned select in one launch, against the same
float32 steps on the host: multiply-adds rounded once (through float64), sums of
an interval's aligned blocks of 16 samples in their order.  The float64 detour of
a multiply-add rounds a second time about once in 2^28, so nearly every knot is
equal; those that are not may differ by what a changed last bit of a gradient
moves them, far less than a step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


def fma(a, b, c):
    return (a.astype(np.float64) * np.float64(b) + c).astype(F)


def steps(orc, J, y, pos, stride, alpha, beta, epochs, lr):
    ns, nk = pos.size, J.size
    u = np.arange(1, ns + 1, dtype=np.int64)
    tgt = (pos.astype(np.float64) - orc.model_line(alpha, beta, (u * stride).astype(np.float64))).astype(F)
    k = np.clip(np.searchsorted(J, u * stride, side="right") - 1, 0, nk - 2)  # an interval holds its first knot
    f = (u * stride - J[k]).astype(F) / (J[k + 1] - J[k]).astype(F)
    w = F(1) - f
    item, at = np.unique(k * ((ns >> 4) + 1) + ((u - 1) >> 4), return_inverse=True)
    q = u - 1 - ((u - 1) >> 4 << 4)
    owner = item // ((ns >> 4) + 1)
    nth = np.arange(item.size) - np.searchsorted(owner, owner)
    m, s = np.zeros(nk, F), np.zeros(nk, F)
    b1, b2, p1, p2 = F(0.9), F(0.999), F(1), F(1)
    scale = F(2) / F(ns)
    for _ in range(epochs):
        e = fma(f, y[k + 1], w * y[k]) - tgt
        sums = []
        for x in (w, f):
            part, full = np.zeros(item.size, F), np.zeros(nk, F)
            for c in range(16):
                i = np.flatnonzero(q == c)
                part[at[i]] = (e[i].astype(np.float64) * x[i] + part[at[i]]).astype(F)
            for c in range(int(nth.max()) + 1):
                i = np.flatnonzero(nth == c)
                full[owner[i]] += part[i]
            sums.append(full)
        g = (sums[0] + np.concatenate([[F(0)], sums[1][:-1]])) * scale
        p1, p2 = p1 * b1, p2 * b2
        m = (np.float64(b1) * m + ((F(1) - b1) * g)).astype(F)
        s = (np.float64(b2) * s + ((F(1) - b2) * g * g)).astype(F)
        y = y - F(lr) * (m / (F(1) - p1)) / (np.sqrt(s / (F(1) - p2)) + F(1e-6))
    return y


@pytest.mark.parametrize("epochs", [1, 10, 11, 27])
def test_steps_in_one_launch(wsfm, orc, ctx, epochs):
    rng = np.random.default_rng(7)
    nb = 1 << 22
    vecs = [rng.random(nb) < d for d in (0.02, 0.5, 0.2)]
    vecs[2][nb // 3:nb // 2] = False
    few = np.zeros(nb, bool)
    few[rng.choice(nb, 40, replace=False)] = True
    vecs.append(few)
    words = []
    for v in vecs:
        words.append(np.append(np.packbits(v, bitorder="little").view(np.uint64), np.uint64(0)))
    dv = [ctx.to_device(w) for w in words]
    par = (16, 4096, 64)
    made = [wsfm.LearnedSelect(ctx, dv, [nb] * len(vecs), wsfm.LselParams(*par, e, 0.5, 512)) for e in (0, epochs)]
    try:
        for b, v in enumerate(vecs):
            (k0, _, _, alpha, beta), (k1, _, _, _, _) = (ls.model(b) for ls in made)
            assert made[1].info(b)["trained"] == 1
            pos = np.flatnonzero(v)[15::16]
            y = steps(orc, k0["j"].astype(np.int64), k0["y"].copy(), pos, 16, alpha, beta, epochs, 0.5)
            print(b, "knots", y.size, "differ", int((y != k1["y"]).sum()), flush=True)
            assert np.array_equal(k0["j"], k1["j"])
            assert (y != k1["y"]).mean() <= 0.01
            assert np.abs(y - k1["y"]).max() <= 0.01 * 0.5 * epochs
    finally:
        for ls in made:
            ls.free()
        for d in dv:
            d.free()


@pytest.mark.parametrize("sizes", [[100, 40000], [1 << 18, 1 << 16, (1 << 17) + 1, 33000] * 6, [1 << 21, 300], [5000]])
def test_plain_structures_of_many_vectors(wsfm, ctx, sizes):
    """Directories and select structures built together (or, of unlike sizes, one by
    one): no ones, all ones, long superblocks, every query against the bits."""
    rng = np.random.default_rng(len(sizes))
    vecs = []
    for b, nb in enumerate(sizes):
        v = rng.random(nb) < (0.5, 0.002, 1.0, 0.0, 0.05, 0.9)[b % 6]
        if b % 6 == 4:
            v[nb // 4:3 * nb // 4] = False
        vecs.append(v)
    dv = []
    for v in vecs:
        w = np.zeros((v.size + 63) // 64 * 8 + 8, np.uint8)
        p = np.packbits(v, bitorder="little")
        w[:p.size] = p
        dv.append(ctx.to_device(w.view(np.uint64)))
    ls = wsfm.LearnedSelect(ctx, dv, sizes)
    try:
        for b, v in enumerate(vecs):
            at = np.flatnonzero(v).astype(np.uint64)
            assert ls.info(b)["ones"] == at.size
            if at.size:
                j = np.unique(np.concatenate([[1, at.size], rng.integers(1, at.size + 1, 3000)])).astype(np.uint64)
                vv = np.full(j.size, b, np.uint32)
                for learned in (False, True):
                    assert np.array_equal(ls.select(vv, j, learned=learned), at[j.astype(np.int64) - 1]), (b, learned)
    finally:
        ls.free()
        for d in dv:
            d.free()
