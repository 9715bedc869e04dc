"""The LDS tail (mg_tail.hpp) at the edges of its per-thread lists: FP64
cycles bitwise the oracle's on lone blocks whose levels hold more cells of
one colour than a thread's registers take (2 x 1024), more ghosts than that,
odd coarsest extents, one-cell extents and the smallest levels, constant and
variable coefficients; several lone blocks in one launch."""
import warnings

import numpy as np
import pytest

from multiflow3d_amd import NotConverged, PressureMultigrid
from multiflow3d_amd import topology as T
from multiflow3d_amd import workloads as W
from oracle.oracle import OracleMG

pytestmark = pytest.mark.gpu

WALLS = [4] * 6
PER = [5] * 6


@pytest.mark.parametrize("n,levels,bc", [
    ((16, 16, 20), 2, T.CHANNEL_BC),   # 2560 cells a colour
    ((64, 24, 2), 2, WALLS),           # 3792 ghosts
    ((12, 20, 28), 3, T.CHANNEL_BC),   # 3 x 5 x 7 at the bottom
    ((8, 4, 4), 3, PER),               # 2 x 1 x 1
    ((6, 2, 10), 2, WALLS),
    ((2, 2, 2), 1, PER),
])
@pytest.mark.parametrize("var", [False, True])
def test_tail_bitwise(n, levels, bc, var):
    grid = T.single_block(list(n), [1.0 / 16, 1.0 / 20, 1.0 / 24], bc)
    f = W.split_blocks(grid, W.global_rhs(grid, W.BASE_SEED + 7, fv_volume=var))
    o = OracleMG(grid.blocks, levels, lsm=var)
    dens = None
    if var:
        dens = [1.0 + 9.0 * (0.5 + 0.5 * W.uniform_pm1(3, 0, f[0].size).reshape(f[0].shape))]
        o.set_density(dens)
    o.coeff()
    p_o, rho_o, _, _ = o.solve(f, 0.0, 3)
    with PressureMultigrid(grid, levels, maxcy=3, eps=0.0, variable_coef=var) as mg:
        if var:
            mg.coeff(dens)
        with warnings.catch_warnings():
            warnings.simplefilter("ignore", NotConverged)
            p_g, res = mg.newsolv_mg(f)
    assert np.array_equal(p_g[0], p_o[0])
    assert np.allclose(res.hist, rho_o, rtol=1e-12, atol=0)


def test_tail_lone_blocks_one_launch():
    # two blocks that do not touch: each its own workgroup, its own lists
    blocks = [T.Block(n=[12, 8, 4], h=[0.1] * 3), T.Block(n=[4, 16, 8], h=[0.1] * 3)]
    f = [W.uniform_pm1(11 + i, 0, b.cells).reshape(b.n[2], b.n[1], b.n[0]) for i, b in enumerate(blocks)]
    f = [a - a.mean() for a in f]
    o = OracleMG(blocks, 3)
    o.coeff()
    p_o, _, _, _ = o.solve(f, 0.0, 3)
    with PressureMultigrid(blocks, 3, maxcy=3, eps=0.0) as mg:
        with warnings.catch_warnings():
            warnings.simplefilter("ignore", NotConverged)
            p_g, _ = mg.newsolv_mg(f)
    for a, b in zip(p_g, p_o):
        assert np.array_equal(a, b)
