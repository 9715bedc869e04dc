"""mf3d_mg_estimate_bytes counts the line smoother's class tables (2 x 3 axes x 16
classes x 48 places a block) where they are larger than the line sequences."""
from multiflow3d_amd import estimate_bytes
from multiflow3d_amd import topology as T


def test_estimate_counts_class_tables():
    grid = T.block_grid([4] * 200, [4], [4], T.CHANNEL_BC, [0.1] * 3)
    for precision, w in (("fp64", 8), ("mixed", 4)):
        kw = dict(precision=precision)
        more = estimate_bytes(grid, 1, smoother=2, **kw) - estimate_bytes(grid, 1, **kw)
        assert more >= 200 * 6 * 16 * 48 * w


def test_estimate_of_ordinary_blocks_is_the_sequences():
    grid = T.block_grid([40] * 80, [10], [25], T.CHANNEL_BC, [0.1] * 3)
    more = estimate_bytes(grid, 1, smoother=2) - estimate_bytes(grid, 1)
    assert more == 80 * 42 * 12 * 27 * 8 * 7   # apr and a of three axes, one scratch
