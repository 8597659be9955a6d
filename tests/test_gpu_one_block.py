"""Trees of at most 8 levels over at most 8192 keys (one block), at the edges of
their chunks and of the size where the multi-block passes take over."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [1, 2, 5, 8])
@pytest.mark.parametrize("n", [1, 7, 63, 64, 65, 1000, 2049, 5003, 8191, 8192, 8193])
@pytest.mark.parametrize("dt", [np.uint8, np.uint16, np.uint32, np.uint64])
def test_one_block(ctx, orc, L, n, dt):
    rng = np.random.default_rng(n + L)
    s = rng.integers(0, 1 << L, n).astype(dt)
    if n % 2:
        s[: n // 2] = (1 << L) - 1  # nodes without keys
    w, nodes = ctx.levels(s, L, with_nodes=True)
    ow, ond = orc.levels_serial(s, L)
    assert np.array_equal(w, ow)
    reached = np.nonzero(ond[:, 5])[0]
    assert np.array_equal(nodes[reached], ond[reached, :5])
    assert np.all(nodes[np.nonzero(ond[:, 5] == 0)[0], 1] == 0)


@pytest.mark.parametrize("n", [100, 5003, 8192])
def test_one_block_bad_symbol(wsfm, ctx, n):
    s = np.zeros(n, np.uint8)
    s[n // 2] = 32
    with pytest.raises(wsfm.WtgError):
        ctx.levels(s, 5)
    ctx.sync()
    s[n // 2] = 31
    w, _ = ctx.levels(s, 5)
    assert int(np.unpackbits(w.view(np.uint8)).sum()) == 5


@pytest.mark.parametrize("n,L", [(20000, 3), (200003, 1), (1 << 20, 8)])
def test_root_tables(ctx, orc, n, L):
    """First-group tables made in one launch (few tiles)."""
    s = np.random.default_rng(n).integers(0, 1 << L, n).astype(np.uint8)
    w, nodes = ctx.levels(s, L, with_nodes=True)
    ow, ond = orc.levels_serial(s, L)
    reached = np.nonzero(ond[:, 5])[0]
    assert np.array_equal(w, ow) and np.array_equal(nodes[reached], ond[reached, :5])
