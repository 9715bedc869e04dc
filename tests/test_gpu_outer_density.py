"""The outer passes with the finest level's coefficients from the density
(MF3D_OUTER_DENSITY=1) against the face arrays (=0), bitwise: tiles of 64 x 8
columns with a remainder and without, the last column of a tile at and beside the
block's end, one plane a chunk and many, walls and periodic faces on every axis,
several blocks; GCR and defect correction, FP64 and mixed."""
import warnings

import numpy as np
import pytest

from multiflow3d_amd import NotConverged, PressureMultigrid
from multiflow3d_amd import topology as T

pytestmark = pytest.mark.gpu

GRIDS = {
    "tile": lambda: T.single_block([64, 8, 4], [1.0 / 16] * 3, T.CHANNEL_BC),
    "one_more_pair": lambda: T.single_block([66, 10, 2], [1.0 / 16, 1.0 / 20, 1.0 / 24], [4] * 6),
    "smallest": lambda: T.single_block([2, 2, 2], [1.0 / 16] * 3, [5, 5, 4, 4, 5, 5]),
    "tiles": lambda: T.single_block([130, 26, 38], [1.0 / 16, 1.0 / 20, 1.0 / 24], [4, 4, 5, 5, 4, 4]),
    "periodic": lambda: T.single_block([62, 16, 70], [1.0 / 16] * 3, [5] * 6),
    "blocks": lambda: T.block_grid([64, 12], [8, 14], [6, 10], T.CHANNEL_BC, [1.0 / 16] * 3),
}


def _solve(grid, dens, f, **kw):
    with PressureMultigrid(grid, 2, variable_coef=True, maxcy=3, eps=0.0, **kw) as mg:
        mg.coeff(dens)
        with warnings.catch_warnings():
            warnings.simplefilter("ignore", NotConverged)
            p, res = mg.newsolv_mg(f)
    return p, res


@pytest.mark.parametrize("name", GRIDS)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("krylov", [False, True])
def test_density_form_bitwise(monkeypatch, name, precision, krylov):
    grid = GRIDS[name]()
    rng = np.random.default_rng(41)
    shapes = [tuple(b.n[::-1]) for b in grid.blocks]
    dens = [np.exp(rng.uniform(0.0, 7.0, s)) for s in shapes]
    f = [rng.standard_normal(s) for s in shapes]
    print(f"[outer density] {name} {precision} krylov={krylov}", flush=True)
    out = []
    for form in "01":
        monkeypatch.setenv("MF3D_OUTER_DENSITY", form)
        out.append(_solve(grid, dens, f, precision=precision, krylov=krylov))
    (pa, ra), (pd, rd) = out
    assert np.array_equal(ra.hist, rd.hist)
    for a, b in zip(pa, pd):
        assert np.isfinite(a).all() and np.array_equal(a, b)


def test_outer_density_switch_error(monkeypatch):
    monkeypatch.setenv("MF3D_OUTER_DENSITY", "2")
    with pytest.raises(Exception, match="MF3D_OUTER_DENSITY"):
        PressureMultigrid(GRIDS["tile"](), 2, variable_coef=True)
