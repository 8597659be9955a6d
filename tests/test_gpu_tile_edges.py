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


@pytest.mark.parametrize("nbits", [1, 64, 511, 512, 513, 32767, 32768, 32769, 65536 + 300, 1 << 20])
@pytest.mark.parametrize("density", [0.0, 0.003, 0.5, 0.997, 1.0])
def test_select_samples_at_tile_edges(ctx, orc, nbits, density):
    """Directory and both sample structures of vectors around the 512-word tiles of
    the sample pass (512 samples of both values a tile, superblock ends among them)."""
    rng = np.random.default_rng(nbits + int(1000 * density))
    bits = rng.random(nbits) < density
    words = np.zeros((nbits + 63) // 64 * 8, np.uint8)
    packed = np.packbits(bits, bitorder="little")
    words[:packed.size] = packed
    words = words.view(np.uint64)
    d = ctx.to_device(words)
    D, s1, s0 = ctx.rank9_select_build(d, nbits)
    try:
        assert np.array_equal(D.get(), orc.rank9_build(words, nbits))
        for s, bit in ((s1, 1), (s0, 0)):
            c, o = s.content(), orc.Select(words, nbits, bit)
            assert c["arg_cnt"] == o.arg_cnt and c["sb"] == o.sb
            assert np.array_equal(c["superblock"], o.superblock[:o.sb])
            assert np.array_equal(c["mini"], o.mini[:o.sb * 64])
            ii = np.unique(np.linspace(1, max(1, o.arg_cnt), 300).astype(np.uint64)) if o.arg_cnt else np.zeros(0, np.uint64)
            if ii.size:
                di = ctx.to_device(ii)
                got = ctx.select_batch(s, d, di)
                assert np.array_equal(got.get(), np.nonzero(bits == bool(bit))[0][ii.astype(np.int64) - 1])
                di.free()
                got.free()
    finally:
        for x in (D, s1, s0, d):
            x.free()
