"""Level-wise trees at the edges of the multi-level passes' tiles (2048 keys, or
4096 for 8-level groups of large inputs), against the oracle's serial build."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1 << 21) - 1, 1 << 21, (1 << 21) + 1, (1 << 21) + 4095, (1 << 21) + 4097])
@pytest.mark.parametrize("skew", [False, True])
def test_byte_tree_wide_tiles(ctx, orc, n, skew):
    rng = np.random.default_rng(n + skew)
    s = rng.integers(0, 256, n).astype(np.uint8)
    if skew:  # long runs of one symbol: leaves that fill whole tiles, others empty
        s[rng.random(n) < 0.97] = 200
    w, nodes = ctx.levels(s, 8, with_nodes=True)
    ow, ond = orc.levels_serial(s, 8)
    assert np.array_equal(w, ow)
    reached = np.nonzero(ond[:, 5])[0]
    assert np.array_equal(nodes[reached], ond[reached, :5])


@pytest.mark.parametrize("levels,extra", [(16, 77), (9, 1), (20, 2047)])
def test_groups_of_several_widths(ctx, orc, levels, extra):
    n = (1 << 23) + extra
    s = np.random.default_rng(levels).integers(0, 1 << levels, n).astype(np.uint32)
    w, _ = ctx.levels(s, levels)
    ow, _ = orc.levels_serial(s, levels, with_nodes=False)
    assert np.array_equal(w, ow)
