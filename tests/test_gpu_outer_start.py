"""The outer iteration's start (k_outer_start): a handle's second solve equals
the first one of a fresh handle, bitwise, so nothing of the first is left in p,
the directions or the residual; on one cell pair, the tile of 64 x 8 columns
with and without a remainder, and several blocks."""
import warnings

import numpy as np
import pytest

from multiflow3d_amd import NotConverged, PressureMultigrid
from multiflow3d_amd import topology as T

pytestmark = pytest.mark.gpu

GRIDS = {
    "smallest": lambda: T.single_block([2, 2, 2], [1.0 / 16] * 3, T.CHANNEL_BC),
    "tile": lambda: T.single_block([64, 8, 32], [1.0 / 16] * 3, [5] * 6),
    "remainder": lambda: T.single_block([66, 10, 34], [1.0 / 16, 1.0 / 20, 1.0 / 24], [4] * 6),
    "blocks": lambda: T.block_grid([64, 12], [8, 14], [6, 10], T.CHANNEL_BC, [1.0 / 16] * 3),
}


def _solve(mg, f):
    with warnings.catch_warnings():
        warnings.simplefilter("ignore", NotConverged)
        return mg.newsolv_mg(f)


@pytest.mark.parametrize("name", GRIDS)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("krylov", [False, True])
def test_second_solve_equals_first(name, precision, krylov):
    grid = GRIDS[name]()
    rng = np.random.default_rng(47)
    fa, fb = ([rng.standard_normal(tuple(b.n[::-1])) for b in grid.blocks] for _ in range(2))
    kw = dict(maxcy=3, eps=0.0, precision=precision, krylov=krylov)
    print(f"[outer start] {name} {precision} krylov={krylov}", flush=True)
    with PressureMultigrid(grid, 2, **kw) as mg:
        _solve(mg, fa)
        p2, r2 = _solve(mg, fb)
    with PressureMultigrid(grid, 2, **kw) as mg:
        p1, r1 = _solve(mg, fb)
    assert r1.hist[0] == 1.0 and np.array_equal(r1.hist, r2.hist)
    for a, b in zip(p1, p2):
        assert np.isfinite(a).all() and np.array_equal(a, b)
