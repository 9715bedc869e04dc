"""Problems near the end of the allocation-free solve's 32 MiB scratch: what is
only there for speed (the LDS tail's lists, the legs' tables, the
line smoother's class tables) is left out where it has no room, so the
numbers of blocks that the solver's fields leave room for are accepted, and
the result is bitwise a handle's."""
import numpy as np
import pytest

from multiflow3d_amd import topology as T
from tests.test_zz_no_alloc import _handle, _noalloc

pytestmark = pytest.mark.gpu

H = [1.0 / 16, 1.0 / 20, 1.0 / 24]


class _Blocks(list):
    """Blocks that do not touch."""

    def __init__(self, n, count):
        super().__init__(T.Block(n=list(n), h=list(H)) for _ in range(count))
        self.blocks = self


def _same(grid, levels, **kw):
    f = np.random.default_rng(83).standard_normal(sum(b.cells for b in grid.blocks))
    print(f"[scratch] {len(grid.blocks)} blocks of {grid.blocks[0].n}, {levels} levels, {kw}", flush=True)
    kw = dict(maxcy=2, eps=0.0, **kw)
    _, p, hist, rmax, k = _noalloc(grid, levels, f, **kw)
    _, ph, hh, rh, kh = _handle(grid, levels, f, **kw)
    assert np.isfinite(p).all() and k == kh == 2 and rmax == rh
    assert np.array_equal(hist, hh[:k + 1]) and np.array_equal(p, ph)


@pytest.mark.parametrize("n,levels,count,precision", [
    ((2, 2, 2), 1, 7013, "fp64"),
    ((2, 2, 2), 1, 8354, "mixed"),
    ((4, 4, 4), 2, 2157, "fp64"),
    ((8, 8, 8), 2, 687, "mixed"),
    ((16, 16, 16), 1, 116, "fp64"),
    ((16, 16, 16), 3, 138, "mixed"),
    ((16, 16, 16), 3, 20, "fp64"),   # room for everything
])
def test_unconnected_blocks_accepted(n, levels, count, precision):
    _same(_Blocks(n, count), levels, precision=precision)


@pytest.mark.parametrize("make,levels,kw", [
    (lambda: T.single_block([8, 8, 6132], H, T.CHANNEL_BC), 2, dict(precision="fp64")),
    (lambda: T.single_block([8, 8, 7478], H, T.CHANNEL_BC), 2, dict(precision="mixed")),
    (lambda: T.block_grid([8] * 93, [8] * 2, [8] * 2, T.CHANNEL_BC, H), 2, dict(precision="fp64", krylov=True)),
    (lambda: T.block_grid([2] * 1252, [2] * 2, [2] * 2, T.CHANNEL_BC, H), 1, dict(precision="fp64", krylov=True)),
], ids=["rod_fp64", "rod_mixed", "grid_gcr", "one_level_gcr"])
def test_legs_without_room(make, levels, kw):
    _same(make(), levels, **kw)


@pytest.mark.parametrize("n,levels,count,precision", [
    ((2, 2, 2), 1, 6195, "mixed"),
    ((4, 4, 4), 2, 1168, "fp64"),
    ((8, 8, 8), 3, 261, "fp64"),
    ((5, 5, 6), 1, 1295, "mixed"),
])
def test_line_smoother_blocks_accepted(n, levels, count, precision):
    _same(T.block_grid([n[0]] * count, [n[1]], [n[2]], [5, 5, 4, 4, 4, 3], H), levels, precision=precision, smoother=2,
          nu_post=1)
