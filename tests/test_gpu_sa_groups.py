"""GPU suffix array at the edges of its refinement windows: groups of equal
prefixes of chosen sizes, against the host's suffix sorter."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(wsfm, ctx, t):
    d = ctx.to_device(t)
    sa = wsfm.suffix_array_gpu(ctx, d, t.size)
    try:
        assert np.array_equal(sa.get(), wsfm.suffix_array(t))
    finally:
        sa.free()
        d.free()


@pytest.mark.parametrize("copies", [2, 3, 64, 511, 512, 513, 1535, 1536, 1537, 2047, 2048, 2049, 4700])
@pytest.mark.parametrize("block,gap", [(30, 1), (24, 40)])
def test_groups_of_copies(wsfm, ctx, copies, block, gap):
    """`copies` of one block, each followed by random letters: every position of
    the block starts a group of that many suffixes, resolved by what follows."""
    rng = np.random.default_rng(copies + block)
    b = rng.integers(65, 69, block).astype(np.uint8)
    parts = [np.concatenate([b, rng.integers(65, 69, gap).astype(np.uint8)]) for _ in range(copies)]
    check(wsfm, ctx, np.concatenate(parts + [np.zeros(1, np.uint8)]))


@pytest.mark.parametrize("n", [2, 25, 64, 1536, 2048, 2049, 5000, 40000])
def test_runs_and_periods(wsfm, ctx, n):
    """One large group that shrinks slowly (a run), and many of them (a period)."""
    check(wsfm, ctx, np.full(n, 66, np.uint8))
    check(wsfm, ctx, np.tile(np.array([66, 67, 66, 65, 66], np.uint8), n // 5 + 1)[:n])


def test_mixed_sizes(wsfm, ctx):
    """Small and large groups side by side, the windows' edges at random places."""
    rng = np.random.default_rng(11)
    blocks = [rng.integers(65, 91, 40).astype(np.uint8) for _ in range(60)]
    pick = rng.choice(60, 9000, p=(w := 1.0 / np.arange(1, 61) ** 1.3) / w.sum())
    parts = [np.concatenate([blocks[k], rng.integers(65, 91, 3).astype(np.uint8)]) for k in pick]
    check(wsfm, ctx, np.concatenate(parts))


@pytest.mark.parametrize("copies", [63, 65, 66, 130, 257, 500, 1000])
@pytest.mark.parametrize("repeats", [1, 3])
def test_groups_sorted_in_a_block(wsfm, ctx, copies, repeats):
    """Groups on either side of the size from which a block is sorted: `copies` of one
    block of letters with few differences among them, so that the ranks h bytes on are
    equal for many suffixes over several rounds; next to small groups."""
    rng = np.random.default_rng(copies + repeats)
    t = np.tile(rng.integers(65, 69, 90).astype(np.uint8), copies)
    at = rng.choice(t.size, copies * repeats // 2 + 1, replace=False)
    t[at] = rng.integers(65, 69, at.size)
    check(wsfm, ctx, np.concatenate([t, rng.integers(65, 69, 3000).astype(np.uint8), np.zeros(1, np.uint8), t[:700]]))
