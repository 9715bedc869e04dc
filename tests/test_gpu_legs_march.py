"""Levels with more 8^3 boxes than the box kernel takes, whose legs march: lone
extents just around one and two tiles of 52 columns and around tiles of 8, 16
and 24 rows, with few and with many rows; block grids with blocks of 8 cells,
smaller than a tile's ring, and uneven ones, walls and periodic faces on every
axis; bitwise the separate kernels' (MF3D_LEGS=0) in FP64, mixed and, on lone
blocks, mixed with variable coefficients.  Then several blocks that do not touch,
of different extents and spacing, in one launch of either kernel: against the
oracle in FP64, and with walls beside periodic faces in y, which no leg takes."""
import warnings

import numpy as np
import pytest
import torch

from multiflow3d_amd import NotConverged, PressureMultigrid
from multiflow3d_amd import topology as T
from oracle.oracle import OracleMG

pytestmark = pytest.mark.gpu

H = [1.0 / 16, 1.0 / 20, 1.0 / 24]
WALLS, PER = [4] * 6, [5] * 6


def _boxes(blocks):
    return sum(int(np.prod([-(-v // 8) for v in b.n])) for b in blocks)


def _solve(blocks, f, dens=None, levels=2, **kw):
    with PressureMultigrid(blocks, levels, maxcy=2, eps=0.0, variable_coef=dens is not None, **kw) as mg:
        if dens is not None:
            mg.coeff(dens)
        with warnings.catch_warnings():
            warnings.simplefilter("ignore", NotConverged)
            return mg.newsolv_mg(f)


def _both(monkeypatch, blocks, form, seed, **kw):
    """The solve with legs and without: the same bits; the one with."""
    rng = np.random.default_rng(seed)
    shapes = [tuple(b.n[::-1]) for b in blocks]
    f = [rng.standard_normal(s) for s in shapes]
    dens = [np.exp(rng.uniform(0.0, 7.0, s)) for s in shapes] if form == "density" else None
    prec = "fp64" if form == "fp64" else "mixed"
    out = []
    for legs in "01":
        monkeypatch.setenv("MF3D_LEGS", legs)
        out.append(_solve(blocks, f, dens, precision=prec, **kw))
    (pa, ra), (pl, rl) = out
    assert np.array_equal(ra.hist, rl.hist)
    for a, b in zip(pa, pl):
        assert np.isfinite(a).all() and np.array_equal(a, b)
    return f, pl, rl


def _marches(blocks):
    assert _boxes(blocks) > 2 * torch.cuda.get_device_properties(0).multi_processor_count


LONE = [
    ((50, 96, 96), WALLS),
    ((52, 96, 96), PER),
    ((54, 96, 96), T.CHANNEL_BC),
    ((102, 72, 96), [4, 4, 5, 5, 5, 5]),
    ((104, 72, 96), [5, 5, 5, 5, 4, 4]),
    ((106, 72, 96), PER),
    ((52, 40, 152), [4, 4, 5, 5, 4, 4]),
    ((104, 104, 40), WALLS),
]


@pytest.mark.parametrize("n,bc", LONE)
@pytest.mark.parametrize("form", ["fp64", "mixed", "density"])
def test_lone_march(monkeypatch, n, bc, form):
    monkeypatch.setenv("MF3D_TAIL", "0")
    grid = T.single_block(list(n), H, bc)
    _marches(grid.blocks)
    print(f"[march] {n} {bc} {form}", flush=True)
    _both(monkeypatch, grid.blocks, form, 89)


GRIDS = {
    "eights_walls": lambda: T.block_grid([8] * 9, [8] * 9, [8] * 8, WALLS, H),
    "eights_periodic": lambda: T.block_grid([8] * 9, [8] * 9, [8] * 8, PER, H),
    "thin_and_wide": lambda: T.block_grid([8, 56, 8], [24, 8, 32], [40, 8, 96], [4, 4, 5, 5, 4, 4], H),
    "around_a_tile": lambda: T.block_grid([52, 8, 54], [8, 40, 8], [64, 24], [5, 5, 4, 4, 4, 4], H),
    "two_tiles": lambda: T.block_grid([104, 50], [16, 24, 32], [64, 48], WALLS, H),
    "few_rows_fp64": lambda: T.block_grid([16] * 4, [24] * 3, [64, 40], [4, 4, 5, 5, 5, 5], H),
}


@pytest.mark.parametrize("name", GRIDS)
@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("nu_pre", [2, 1])
def test_block_march(monkeypatch, name, form, nu_pre):
    grid = GRIDS[name]()
    _marches(grid.blocks)
    print(f"[block march] {name} {form} V({nu_pre},2)", flush=True)
    _both(monkeypatch, grid.blocks, form, 97, nu_pre=nu_pre)


SIZES = {"boxes": [(16, 8, 24), (24, 16, 8)], "march": [(56, 64, 48), (40, 80, 72), (104, 16, 40)]}


def _apart(size, faces):
    """Blocks that do not touch, spacing of their own; faces: one set of codes a block."""
    return [T.Block(n=list(n), h=[h * (1.0 + 0.25 * i) for h in H], bc=list(bc))
            for i, (n, bc) in enumerate(zip(SIZES[size], faces))]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("bc", [WALLS, T.CHANNEL_BC, PER], ids=["walls", "channel", "periodic"])
def test_unconnected_blocks(monkeypatch, size, bc):
    monkeypatch.setenv("MF3D_TAIL", "0")
    blocks = _apart(size, [bc] * 3)
    if size == "march":
        _marches(blocks)
    print(f"[apart] {size} {bc}", flush=True)
    f, p, _ = _both(monkeypatch, blocks, "fp64", 101)
    o = OracleMG(blocks, 2)
    o.coeff()
    p_o, _, _, _ = o.solve(f, 0.0, 2)
    for a, b in zip(p, p_o):
        assert np.array_equal(a, b)
    _both(monkeypatch, blocks, "mixed", 103)
    _both(monkeypatch, blocks, "density", 107)


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("form", ["fp64", "mixed", "density"])
def test_unconnected_blocks_with_mixed_y_faces(monkeypatch, size, form):
    monkeypatch.setenv("MF3D_TAIL", "0")
    print(f"[apart, mixed y] {size} {form}", flush=True)
    _both(monkeypatch, _apart(size, [WALLS, PER, T.CHANNEL_BC]), form, 109)
