"""One V-cycle on a caller's potential whose ghosts are not those of its interior
(mgkcyc): without pre-sweeps the prolongation and the first post-sweep read them
as they are, so level 0 runs no up leg there; FP64 bitwise the oracle's, ghosts
included, mixed bitwise the separate kernels' (MF3D_LEGS=0); box and march sizes,
lone blocks and a block grid, walls and periodic faces.  The same for a cycle that
the LDS tail runs whole and for the line smoother, whose kernels read ghosts too."""
import numpy as np
import pytest

from multiflow3d_amd import PressureMultigrid
from multiflow3d_amd import topology as T
from oracle.oracle import OracleMG

pytestmark = pytest.mark.gpu

H = [1.0 / 16, 1.0 / 20, 1.0 / 24]
GRIDS = {
    "boxes_periodic": lambda: T.single_block([32, 16, 24], H, [5] * 6),
    "boxes_channel": lambda: T.single_block([16, 32, 16], H, T.CHANNEL_BC),
    "march_periodic": lambda: T.single_block([72, 64, 72], H, [5] * 6),
    "blocks_channel": lambda: T.block_grid([16, 24], [8, 16], [24, 8], T.CHANNEL_BC, H),
    "blocks_march": lambda: T.block_grid([8] * 9, [8] * 9, [8] * 8, [4, 4, 5, 5, 5, 5], H),
}


@pytest.mark.parametrize("name", GRIDS)
@pytest.mark.parametrize("nu_pre", [0, 1, 2])
def test_cycle_from_any_ghosts(monkeypatch, name, nu_pre):
    monkeypatch.setenv("MF3D_TAIL", "0")
    grid = GRIDS[name]()
    rng = np.random.default_rng(113)
    f = [rng.standard_normal(tuple(b.n[::-1])) for b in grid.blocks]
    pp = [rng.standard_normal(tuple(v + 2 for v in b.n[::-1])) for b in grid.blocks]
    o = OracleMG(grid.blocks, 2, nu_pre=nu_pre, nu_post=2)
    o.coeff()
    want = o.vcycle(f, [a.copy() for a in pp])
    print(f"[cycle from ghosts] {name} V({nu_pre},2)", flush=True)

    def run(precision):
        got = [a.copy() for a in pp]
        with PressureMultigrid(grid, 2, nu_pre=nu_pre, nu_post=2, precision=precision) as mg:
            return mg.mgkcyc(f, got)

    for a, b in zip(run("fp64"), want):
        assert np.array_equal(a, b)
    mixed = run("mixed")
    monkeypatch.setenv("MF3D_LEGS", "0")
    for a, b in zip(mixed, run("mixed")):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("make,levels,smoother", [
    (lambda: T.single_block([16, 16, 16], H, [5] * 6), 3, 3),
    (lambda: T.single_block([16, 8, 20], H, T.CHANNEL_BC), 2, 3),
    (lambda: T.single_block([12, 20, 8], H, [5, 5, 4, 4, 5, 5]), 1, 2),
    (lambda: T.block_grid([8, 12], [10], [6], [5, 5, 4, 4, 4, 3], H), 2, 2),
], ids=["tail_periodic", "tail_channel", "lines", "lines_blocks"])
@pytest.mark.parametrize("nu_pre", [0, 1])
def test_tail_and_lines_from_any_ghosts(make, levels, smoother, nu_pre):
    grid = make()
    rng = np.random.default_rng(127)
    f = [rng.standard_normal(tuple(b.n[::-1])) for b in grid.blocks]
    pp = [rng.standard_normal(tuple(v + 2 for v in b.n[::-1])) for b in grid.blocks]
    o = OracleMG(grid.blocks, levels, nu_pre=nu_pre, nu_post=2, smoother=smoother)
    o.coeff()
    want = o.vcycle(f, [a.copy() for a in pp])
    got = [a.copy() for a in pp]
    with PressureMultigrid(grid, levels, nu_pre=nu_pre, nu_post=2, smoother=smoother) as mg:
        mg.mgkcyc(f, got)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
