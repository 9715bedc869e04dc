"""The one-launch legs (k_leg) against the oracle, FP64 bitwise, and in FP32
against the same cycle with sweeps, restriction and prolongation apart
(MF3D_LEGS=0), bitwise too: extents around the tile (52 x 8, 52 x 16 and
52 x 24 cells), the smallest extent (8), levels that leave compute units idle
and one (106 x 98 x 96) that does not, walls and periodic faces on every axis,
the LDS tail off so that every level above the coarsest runs them, and the
up leg only (V(1,2)) or neither (V(2,1))."""
import warnings

import numpy as np
import pytest

from multiflow3d_amd import NotConverged, PressureMultigrid
from multiflow3d_amd import topology as T
from multiflow3d_amd import workloads as W
from oracle.oracle import OracleMG

pytestmark = pytest.mark.gpu

WALLS, PER = [4] * 6, [5] * 6
SHAPES = [
    ((8, 8, 8), 2, T.CHANNEL_BC),
    ((16, 8, 24), 2, PER),
    ((52, 16, 12), 2, T.CHANNEL_BC),
    ((56, 24, 8), 3, PER),
    ((104, 26, 10), 2, [5, 5, 5, 5, 4, 4]),
    ((54, 48, 34), 2, WALLS),
    ((40, 20, 96), 3, [4, 4, 5, 5, 5, 5]),
    ((64, 64, 64), 4, PER),
    ((106, 98, 96), 2, [5, 5, 4, 4, 5, 5]),
]


def _solve(grid, levels, f, cycles, **kw):
    with PressureMultigrid(grid, levels, maxcy=cycles, eps=0.0, **kw) as mg:
        with warnings.catch_warnings():
            warnings.simplefilter("ignore", NotConverged)
            p, res = mg.newsolv_mg(f)
    return p[0], res.hist


@pytest.mark.parametrize("n,levels,bc", SHAPES)
@pytest.mark.parametrize("nu", [(2, 2), (2, 1), (1, 2)])
def test_legs_bitwise(monkeypatch, n, levels, bc, nu):
    monkeypatch.setenv("MF3D_TAIL", "0")
    grid = T.single_block(list(n), [1.0 / 16, 1.0 / 20, 1.0 / 24], bc)
    f = W.split_blocks(grid, W.global_rhs(grid, W.BASE_SEED + 13))
    o = OracleMG(grid.blocks, levels, nu_pre=nu[0], nu_post=nu[1])
    o.coeff()
    p_o, rho_o, _, _ = o.solve(f, 0.0, 3)
    print(f"[legs] {n} {nu}", flush=True)
    p, hist = _solve(grid, levels, f, 3, nu_pre=nu[0], nu_post=nu[1])
    assert np.array_equal(p, p_o[0])
    assert np.allclose(hist, rho_o, rtol=1e-12, atol=0)
    pm, hm = _solve(grid, levels, f, 3, nu_pre=nu[0], nu_post=nu[1], precision="mixed")
    monkeypatch.setenv("MF3D_LEGS", "0")
    pa, ha = _solve(grid, levels, f, 3, nu_pre=nu[0], nu_post=nu[1], precision="mixed")
    assert np.array_equal(pm, pa) and np.array_equal(hm, ha)


def test_legs_switch_error(monkeypatch):
    monkeypatch.setenv("MF3D_LEGS", "2")
    with pytest.raises(Exception, match="MF3D_LEGS"):
        PressureMultigrid(T.single_block(16, [1 / 16] * 3, T.CHANNEL_BC), 2)
