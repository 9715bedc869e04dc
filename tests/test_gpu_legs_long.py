"""Legs of lone levels with too many 8^3 boxes for the box kernel and one axis
of 8 cells, marched: along x, y and z, against the separate kernels
(MF3D_LEGS=0), bitwise, in FP64, mixed and mixed with variable coefficients."""
import warnings

import numpy as np
import pytest

from multiflow3d_amd import NotConverged, PressureMultigrid
from multiflow3d_amd import topology as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(8, 168, 200), (168, 8, 208), (200, 176, 8)])
@pytest.mark.parametrize("bc", [[5] * 6, [4] * 6])
@pytest.mark.parametrize("form", ["fp64", "mixed", "density"])
def test_long_levels_bitwise(monkeypatch, n, bc, form):
    grid = T.single_block(list(n), [1.0 / 16, 1.0 / 20, 1.0 / 24], bc)
    rng = np.random.default_rng(67)
    f = [rng.standard_normal(n[::-1])]
    dens = [np.exp(rng.uniform(0.0, 7.0, n[::-1]))] if form == "density" else None
    print(f"[long legs] {n} {bc[0]} {form}", flush=True)
    out = []
    for legs in "01":
        monkeypatch.setenv("MF3D_LEGS", legs)
        with PressureMultigrid(grid, 2, maxcy=2, eps=0.0, precision="fp64" if form == "fp64" else "mixed",
                               variable_coef=dens is not None) as mg:
            if dens is not None:
                mg.coeff(dens)
            with warnings.catch_warnings():
                warnings.simplefilter("ignore", NotConverged)
                out.append(mg.newsolv_mg(f))
    (pa, ra), (pl, rl) = out
    assert np.isfinite(pa[0]).all() and np.array_equal(pa[0], pl[0]) and np.array_equal(ra.hist, rl.hist)
