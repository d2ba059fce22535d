"""What vt_free_map_used says of a frame's statistics, at every size from the
smallest world (16^3, one region) on: 1 exactly when they count the steps
executed -- fewer than traceMap's wherever a ray crosses the empty world -- and
0 when they are traceMap's, the oracle's counts.  Empty worlds, worlds with a
voxel in a corner (free regions in the other octants from 32^3 on), full
floors, before and after an edit that empties them."""
import numpy as np
import pytest

import oracle_ffi as O
import vt
from test_gpu_freemap import OFF, ON, render_free
from vt import scenes as S

pytestmark = pytest.mark.gpu

W, H = 40, 32


def steps(ctx, w, cam, flags):
    import torch
    f = vt.Frame.alloc(W, H, stats=True)
    prm = vt.params(W, H, 600, 600, S.SUN, flags)
    vt.render(ctx, w, cam, f, prm)
    torch.cuda.synchronize()
    d = f.stats_dict()
    return vt.free_map_used(w, f, prm), d["primary_steps"] + d["shadow_steps"]


@pytest.mark.parametrize("kind", ["empty", "corner", "floor"])
@pytest.mark.parametrize("n", [16, 32, 64, 128])
def test_statistics_are_what_the_rule_says(ctx, n, kind):
    grid, pal = np.zeros((n, n, n), np.uint8), S.palette()
    if kind == "corner":
        grid[0, 0, 0] = 4
    elif kind == "floor":
        grid[:, 0, :] = 3
    w = vt.World.dense(ctx, grid, pal)
    cam = vt.look_at((n / 2 + 0.3, n * 0.7, -0.4 * n), (n / 2, n * 0.3, n / 2), 70.0)
    for turn in range(2):
        o = O.render(O.DenseWorld(grid, pal), cam, W, H, 600, 600, S.SUN)
        ref = int(np.sum(o["steps"] & 0xFFFF) + np.sum(o["steps"] >> 16))
        assert ref > 0
        for flags in (0, OFF, ON):
            used, got = steps(ctx, w, cam, flags)
            assert used == (flags == ON and (n > 16 or not grid.any())), (n, kind, turn, flags)
            assert got < ref if used else got == ref, (n, kind, turn, flags, got, ref)
            r = render_free(ctx, w, cam, W, H, 600, 600, S.SUN, flags, gbuffer=False)
            assert np.array_equal(r["hits"], o["hits"])
        z, y, x = np.nonzero(grid)
        if len(x):
            w.set_voxels(np.stack([x, y, z], 1), np.zeros(len(x), np.uint32))
        grid[:] = 0
    w.close()
