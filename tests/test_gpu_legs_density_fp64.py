"""The box kernel's legs with variable coefficients in FP64 against the same
cycle with sweeps, restriction and prolongation apart (MF3D_LEGS=0), bitwise: the
smallest extent (8), remainders of a box (8 cells), walls and periodic faces
(one-sided at the block's edge) on every axis, a finest level with too many
boxes above one with few, both coarse operators."""
import warnings

import numpy as np
import pytest

from multiflow3d_amd import NotConverged, PressureMultigrid
from multiflow3d_amd import topology as T

pytestmark = pytest.mark.gpu

SHAPES = [
    ((8, 8, 8), 2, T.CHANNEL_BC),
    ((16, 8, 24), 2, [5] * 6),
    ((10, 20, 12), 2, [4] * 6),
    ((24, 26, 10), 2, [5, 5, 4, 4, 4, 4]),
    ((80, 64, 72), 4, [5, 5, 4, 4, 5, 5]),
]


@pytest.mark.parametrize("n,levels,bc", SHAPES)
@pytest.mark.parametrize("nu,coarse_op", [((2, 2), "face"), ((2, 2), "reference"), ((1, 2), "face")])
def test_density_legs_fp64_bitwise(monkeypatch, n, levels, bc, nu, coarse_op):
    monkeypatch.setenv("MF3D_TAIL", "0")
    grid = T.single_block(list(n), [1.0 / 16, 1.0 / 20, 1.0 / 24], bc)
    rng = np.random.default_rng(71)
    dens = [np.exp(rng.uniform(0.0, 7.0, n[::-1]))]
    f = [rng.standard_normal(n[::-1])]
    print(f"[density legs fp64] {n} {nu} {coarse_op}", flush=True)
    out = []
    for legs in "01":
        monkeypatch.setenv("MF3D_LEGS", legs)
        with PressureMultigrid(grid, levels, maxcy=3, eps=0.0, variable_coef=True, nu_pre=nu[0], nu_post=nu[1],
                               coarse_op=coarse_op) as mg:
            mg.coeff(dens)
            with warnings.catch_warnings():
                warnings.simplefilter("ignore", NotConverged)
                out.append(mg.newsolv_mg(f))
    (pa, ra), (pl, rl) = out
    assert np.isfinite(pa[0]).all() and np.array_equal(pa[0], pl[0]) and np.array_equal(ra.hist, rl.hist)
