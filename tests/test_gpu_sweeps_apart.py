"""The sweep, prolongation and exchange kernels with the one-launch legs off
(MF3D_LEGS=0), where the switches between their forms decide every level: pinned
march depths and the zero-start march against the one-pass 3-D tiles, the fused
prolongation against the separate one, each layout switch against the default, in
both precisions; FP64 cycles bitwise the oracle's."""
import warnings

import numpy as np
import pytest

from multiflow3d_amd import NotConverged
from oracle.oracle import OracleMG
from tests.cases import case, inputs
from tests.test_gpu_parity import _gpu

pytestmark = pytest.mark.gpu

NAMES = ["single64_L5", "multi_uneven_L3", "periodic_multi_L3", "neumann_L4"]


@pytest.fixture(autouse=True)
def _legs_off(monkeypatch):
    monkeypatch.setenv("MF3D_LEGS", "0")


def _run(name, f, precision, cycles=3):
    grid, L, _ = case(name)
    with _gpu(grid, L, False, None, maxcy=cycles, eps=0.0, precision=precision) as mg:
        with warnings.catch_warnings():
            warnings.simplefilter("ignore", NotConverged)
            return mg.newsolv_mg(f)


def _same(a, b, rtol=0):
    np.testing.assert_allclose(a[1].hist, b[1].hist, rtol=rtol, atol=0)
    for x, y in zip(a[0], b[0]):
        assert np.isfinite(x).all() and np.array_equal(x, y)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("zero", ["1", "0"], ids=["zero_march", "zero_full"])
@pytest.mark.parametrize("tz", ["2", "4", "6", "16"])
@pytest.mark.parametrize("name", NAMES)
def test_march_depths(name, tz, zero, precision, monkeypatch):
    grid, _, _ = case(name)
    f, _ = inputs(grid, False, seed=29)
    monkeypatch.setenv("MF3D_ZERO_SWEEP", zero)
    monkeypatch.setenv("MF3D_SWEEP_3D", "1")
    tiles = _run(name, f, precision)
    monkeypatch.setenv("MF3D_SWEEP_3D", "0")
    monkeypatch.setenv("MF3D_SWEEP_TZ", tz)
    _same(tiles, _run(name, f, precision))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("name", ["single32_L5", *NAMES])
def test_fused_prolongation(name, precision, monkeypatch):
    grid, _, _ = case(name)
    f, _ = inputs(grid, False, seed=31)
    monkeypatch.setenv("MF3D_SWEEP_3D", "1")
    fused = _run(name, f, precision)
    monkeypatch.setenv("MF3D_FUSE_PROLONG", "0")
    _same(fused, _run(name, f, precision))


@pytest.mark.parametrize("var,val", [("MF3D_SWEEP_3D", "1"), ("MF3D_SWEEP_3D", "0"), ("MF3D_ZERO_SWEEP", "0"),
                                     ("MF3D_OWN_GHOSTS", "0"), ("MF3D_XCD_ORDER", "0"), ("MF3D_TAIL", "0"),
                                     ("MF3D_AUTOTUNE", "0")])
@pytest.mark.parametrize("name", NAMES)
def test_switches(name, var, val, monkeypatch):
    grid, L, _ = case(name)
    f, _ = inputs(grid, False, seed=37)
    default = {p: _run(name, f, p) for p in ("fp64", "mixed")}
    monkeypatch.setenv(var, val)
    # the residual norm is summed over workgroups, whose order this one changes
    rtol = 1e-12 if var == "MF3D_XCD_ORDER" else 0
    for p in default:
        _same(default[p], _run(name, f, p), rtol)
    o = OracleMG(grid.blocks, L)
    o.coeff()
    p_o, _, _, _ = o.solve(f, 0.0, 3)
    for a, b in zip(default["fp64"][0], p_o):
        assert np.array_equal(a, b)
