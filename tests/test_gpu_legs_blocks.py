"""The one-launch legs (k_leg) on grids of several blocks against the oracle,
FP64 bitwise, and in FP32 against the same cycle with sweeps, restriction and
prolongation apart (MF3D_LEGS=0), bitwise too: blocks smaller than a tile's ring
and tile (8 cells) and larger, uneven extents, one block periodic onto itself
beside others along another axis, two blocks that are each other's neighbours on
both sides, walls and periodic faces on every axis, levels that leave compute
units idle and one that does not.  An L of three blocks, whose walls end at a
face, takes the separate kernels: the same with and without the legs."""
import warnings

import numpy as np
import pytest

from multiflow3d_amd import NotConverged, PressureMultigrid
from multiflow3d_amd import topology as T
from multiflow3d_amd import workloads as W
from oracle.oracle import OracleMG

pytestmark = pytest.mark.gpu

H = [1.0 / 16, 1.0 / 20, 1.0 / 24]
WALLS, PER = [4] * 6, [5] * 6


def _ell():
    g = T.block_grid([16, 24], [8, 16], [8], WALLS, H)
    g.blocks[1].nbr[3] = g.blocks[2].nbr[1] = -1
    g.blocks = g.blocks[:3]
    return g


GRIDS = {
    "eight_channel": (lambda: T.block_grid([16, 24], [8, 16], [24, 8], T.CHANNEL_BC, H), 2),
    "eight_walls": (lambda: T.block_grid([8, 8], [8, 8], [8, 8], WALLS, H), 2),
    "eight_periodic": (lambda: T.block_grid([8, 60], [24, 8], [8, 16], PER, H), 2),
    "row_x": (lambda: T.block_grid([16, 8, 56], [24], [16], [4, 4, 5, 5, 5, 5], H), 2),
    "row_y": (lambda: T.block_grid([64], [8, 16, 8], [16], [5, 5, 4, 4, 4, 4], H), 2),
    "row_z": (lambda: T.block_grid([16], [16], [8, 8, 24], [5, 5, 5, 5, 5, 5], H), 2),
    "three_levels": (lambda: T.block_grid([48, 32], [32, 48], [32, 64], T.CHANNEL_BC, H), 4),
    "large": (lambda: T.block_grid([104, 64], [80, 64], [64, 96], PER, H), 2),
}


def _solve(grid, levels, f, **kw):
    with PressureMultigrid(grid, levels, maxcy=3, eps=0.0, **kw) as mg:
        with warnings.catch_warnings():
            warnings.simplefilter("ignore", NotConverged)
            return mg.newsolv_mg(f)


@pytest.mark.parametrize("name", GRIDS)
@pytest.mark.parametrize("nu", [(2, 2), (1, 2)])
def test_block_legs_bitwise(monkeypatch, name, nu):
    make, levels = GRIDS[name]
    grid = make()
    rng = np.random.default_rng(53)
    f = [rng.standard_normal(tuple(b.n[::-1])) for b in grid.blocks]
    o = OracleMG(grid.blocks, levels, nu_pre=nu[0], nu_post=nu[1])
    o.coeff()
    p_o, rho_o, _, _ = o.solve(f, 0.0, 3)
    print(f"[block legs] {name} {nu}", flush=True)
    kw = dict(nu_pre=nu[0], nu_post=nu[1])
    p, res = _solve(grid, levels, f, **kw)
    assert np.allclose(res.hist, rho_o, rtol=1e-12, atol=0)
    for a, b in zip(p, p_o):
        assert np.array_equal(a, b)
    pm, rm = _solve(grid, levels, f, precision="mixed", **kw)
    monkeypatch.setenv("MF3D_LEGS", "0")
    pa, ra = _solve(grid, levels, f, precision="mixed", **kw)
    assert np.array_equal(rm.hist, ra.hist)
    for a, b in zip(pm, pa):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_ell_takes_separate_kernels(monkeypatch, precision):
    grid = _ell()
    rng = np.random.default_rng(59)
    f = [rng.standard_normal(tuple(b.n[::-1])) for b in grid.blocks]
    p, r = _solve(grid, 2, f, precision=precision)
    monkeypatch.setenv("MF3D_LEGS", "0")
    pa, ra = _solve(grid, 2, f, precision=precision)
    assert np.array_equal(r.hist, ra.hist)
    for a, b in zip(p, pa):
        assert np.array_equal(a, b)
