"""wt_huff bits at the edges of the tile emit: segment sizes, alphabets around its
smallest tree, codes at and past its longest; against the oracle's shape and bits."""
import numpy as np
import pytest

from test_gpu_huff import check_shape, fib_text

pytestmark = pytest.mark.gpu


def check(ctx, orc, t):
    d = ctx.to_device(t)
    wt = ctx.huff_build(d)
    try:
        oh = orc.Huff(t)
        check_shape(wt, oh)
        words = wt.words()
        assert np.array_equal(words[:(oh.nbits + 63) // 64], oh.words) and words[-1] == 0
        assert np.array_equal(wt.directory(), oh.D)
    finally:
        wt.free()
        d.free()


@pytest.mark.parametrize("sigma", [17, 18, 19, 129, 256])
@pytest.mark.parametrize("n", [300, 4095, 4096, 4097, 12289, 100003])
def test_tile_edges(ctx, orc, sigma, n):
    rng = np.random.default_rng(n + sigma)
    p = 1.0 / np.arange(1, sigma + 1)
    t = rng.choice(sigma, n, p=p / p.sum()).astype(np.uint8)
    t[:sigma] = np.arange(sigma)  # every symbol occurs
    check(ctx, orc, t)


@pytest.mark.parametrize("symbols", [18, 23, 24, 25, 26])
def test_code_lengths(ctx, orc, symbols):
    """Fibonacci counts: codes of symbols - 1 bits (23 is the tile emit's longest)."""
    check(ctx, orc, fib_text(np.random.default_rng(symbols), symbols))


def test_segment_of_one_symbol(ctx, orc):
    """Segments whose keys all take one path, next to uniform ones."""
    rng = np.random.default_rng(5)
    t = np.concatenate([np.full(9000, 7, np.uint8), rng.integers(0, 256, 8192).astype(np.uint8), np.full(5000, 200, np.uint8)])
    check(ctx, orc, t)
