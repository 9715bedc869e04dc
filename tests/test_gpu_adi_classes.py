"""The constant-coefficient ADI sweep (k_adi_cls) at the edges of its rule and
of its chunks, FP64 bitwise the oracle's: lines of one cell, of whole and
broken groups of 4 and 8, extents of 48 (its longest line) and 49 (the sweep
it leaves to), one, two and five cells a thread, every wall / periodic /
neighbour combination of the line classes, single-cell axes."""
import warnings

import numpy as np
import pytest

from multiflow3d_amd import NotConverged, PressureMultigrid
from multiflow3d_amd import topology as T
from multiflow3d_amd import workloads as W
from oracle.oracle import OracleMG

pytestmark = pytest.mark.gpu

CASES = [
    ([40, 40], [10], [25], [5, 5, 4, 4, 4, 3]),       # the shipped deck's blocks
    ([17], [9], [8], [4] * 6),
    ([16], [7], [24], [5] * 6),
    ([48], [12], [5], T.CHANNEL_BC),                  # two cells a thread
    ([5], [48], [31], [4, 4, 5, 5, 4, 4]),            # five
    ([49], [6], [5], [4] * 6),                        # a line too long: the other sweep
    ([1], [4], [3], [4] * 6),
    ([3], [1], [33], [5, 5, 4, 4, 5, 5]),
    ([2, 3], [12, 4], [1], [4, 4, 4, 4, 5, 5]),
    ([6, 11], [5], [4, 9], [5, 5, 4, 4, 5, 5]),
]


@pytest.mark.parametrize("ex,ey,ez,bc", CASES)
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_adi_classes(ex, ey, ez, bc, prec):
    grid = T.block_grid(ex, ey, ez, bc, [0.05, 0.04, 0.06])
    f = W.split_blocks(grid, W.global_rhs(grid, W.BASE_SEED + 9))
    o = OracleMG(grid.blocks, 1, smoother=2, nu_pre=2, nu_post=1)
    o.coeff()
    p_o, rho_o, _, _ = o.solve(f, 0.0, 4)
    with PressureMultigrid(grid, 1, smoother=2, nu_pre=2, nu_post=1, maxcy=4, eps=0.0, precision=prec) as mg:
        with warnings.catch_warnings():
            warnings.simplefilter("ignore", NotConverged)
            p_g, res = mg.newsolv_mg(f)
    if prec == "fp64":
        for a, b in zip(p_g, p_o):
            assert np.array_equal(a, b)
        assert np.allclose(res.hist, rho_o, rtol=1e-12, atol=0)
    else:
        # each cycle's correction carries FP32 rounding (2^-24 a step over a few
        # hundred dependent steps), relative to the correction
        scale = max(np.abs(b).max() for b in p_o)
        assert max(np.abs(a - b).max() for a, b in zip(p_g, p_o)) <= 1e-4 * scale
