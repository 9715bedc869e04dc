"""Host arrays of the velocity form packed by several threads (fields of 3 MiB
and more) against the device-resident call, bitwise: one and two ghost layers,
a block of one piece beside blocks of many, and a second call on the same handle."""
import numpy as np
import pytest
import torch

from multiflow3d_amd import PressureMultigrid
from multiflow3d_amd import topology as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ghost", [1, 2])
@pytest.mark.parametrize("ex,ey,ez", [([64], [48], [160]), ([60, 4], [64, 36], [32, 48])])
def test_host_fields_match_device(ghost, ex, ey, ez):
    grid = T.block_grid(ex, ey, ez, T.CHANNEL_BC, [1.0 / 64] * 3)
    shapes = [tuple(d + 2 * ghost for d in b.n[::-1]) for b in grid.blocks]
    rng = np.random.default_rng(61)
    kw = dict(maxcy=2, eps=0.0, ghost=ghost)
    print(f"[host fields] {ex} {ey} {ez} ghost {ghost}", flush=True)
    with PressureMultigrid(grid, 2, **kw) as mg:
        for _ in range(2):
            fields = [[rng.standard_normal(s) for s in shapes] for _ in range(7)]
            dev = [torch.from_numpy(np.concatenate([a.ravel() for a in q])).cuda() for q in fields]
            torch.cuda.synchronize()
            h = mg.newsolv(*fields, 0.01, 1.0, 0.0, warn=False)
            d = mg.newsolv_device([t.data_ptr() for t in dev], 0.01, 1.0, 0.0, warn=False)
            torch.cuda.synchronize()
            assert np.array_equal(h.hist, d.hist)
            for q, t in zip(fields, dev):
                assert np.array_equal(np.concatenate([a.ravel() for a in q]), t.cpu().numpy())
