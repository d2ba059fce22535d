"""The clearance map after edits, read by the frames that are compared:
VT_FLAG_FREE_MAP_ON, so that no rule on the world's openness leaves it aside.
Frames must be the oracle's, the free-region map a fresh world's, and on dense
worlds the steps that the statistics count with that flag a fresh world's too:
they depend on every byte of the map that a ray reads."""
import numpy as np
import pytest

import brickmap_util as BU
import oracle_ffi as O
import vt
from test_gpu_clear import check
from test_gpu_freemap import ON, SUNS, render_free
from vt import scenes as S

pytestmark = pytest.mark.gpu

W, H, CAP = 64, 48, 700


def fresh(ctx, layout, grid):
    if layout == "dense":
        return vt.World.dense(ctx, grid, S.palette())
    return vt.World.brickmap(ctx, *BU.embedding_a(grid, S.palette()))


def executed(ctx, w, cam, sun):
    import torch
    f = vt.Frame.alloc(W, H, stats=True)
    vt.render(ctx, w, cam, f, vt.params(W, H, CAP, CAP, sun, ON))
    torch.cuda.synchronize()
    return f.stats.cpu().tolist()


def equals_fresh_world(ctx, layout, w, grid, label):
    n = grid.shape[0]
    f, ow = fresh(ctx, layout, grid), O.DenseWorld(grid, S.palette())
    a, av = w.read_free_map()
    b, bv = f.read_free_map()
    assert av and bv and np.array_equal(a, b), f"{layout} {label}: free-region map"
    for k, (eye, at) in enumerate((((-0.3, 0.8, -0.4), (0.5, 0.3, 0.5)),
                                   ((0.9, 0.9, 0.8), (0.1, 0.2, 0.2)),
                                   ((0.5, 0.05, 1.3), (0.5, 0.6, 0.1)))):
        cam = vt.look_at(*(tuple(n * c for c in p) for p in (eye, at)), 70.0)
        o = O.render(ow, cam, W, H, CAP, CAP, SUNS[k])
        check(render_free(ctx, w, cam, W, H, CAP, CAP, SUNS[k], ON, gbuffer=False), o,
              f"{layout} {label}: camera {k}")
        if layout == "dense":
            assert executed(ctx, w, cam, SUNS[k]) == executed(ctx, f, cam, SUNS[k]), (label, k)
    f.close()


def apply(w, grid, xyz, val):
    w.set_voxels(xyz, val)
    for (x, y, z), v in zip(xyz, val):  # in order: the last write wins
        grid[z, y, x] = v


@pytest.mark.parametrize("layout", ["dense", "reference"])
def test_lists_in_any_order(ctx, layout):
    """Lists that come back to the same 4^3 bricks again and again, setting
    some of their voxels and clearing others, in the staging and above it."""
    n = 64
    rng = np.random.default_rng(11)
    grid = np.zeros((n, n, n), np.uint8)
    grid[:, :2] = 3
    w = fresh(ctx, layout, grid)
    for count in (60, 5000, 16384, 16385, 30000):
        corner = rng.integers(0, n - 6, (6, 3))
        xyz = corner[rng.integers(0, 6, count)] + rng.integers(0, 6, (count, 3))
        val = rng.integers(0, 3, count) * (rng.random(count) < 0.3)
        apply(w, grid, xyz.astype(np.uint32), val.astype(np.uint32))
        equals_fresh_world(ctx, layout, w, grid, f"{count} edits")
    w.close()


@pytest.mark.parametrize("n", [32, 128])
@pytest.mark.parametrize("layout", ["dense", "reference"])
def test_cleared_and_refilled(ctx, layout, n):
    """2^3 sub-blocks filled, cleared in part, cleared whole and filled again,
    alone in clear space, next to other things, in the corners of the grid and
    of the map's 8^3 cells, one by one and many at a time."""
    rng = np.random.default_rng([n, 5])
    grid = np.zeros((n, n, n), np.uint8)
    grid[:, :2] = 3
    grid[n // 2, :n // 3, n // 2] = 4
    w = fresh(ctx, layout, grid)
    sub = np.stack([v.ravel() for v in np.mgrid[0:2, 0:2, 0:2]], 1)
    lows = np.vstack([[0, n - 2, 0], [n - 2, n - 2, n - 2], [6, 14, 6], [8, 16, 8],
                      [n // 2, n // 3, n // 2], 2 * rng.integers(1, n // 2, (6, 3))])
    all_of = (lows[:, None] + sub[None]).reshape(-1, 3).astype(np.uint32)
    steps = [("filled", all_of, 5), ("thinned", all_of[::2], 0), ("cleared", all_of, 0)]
    for k, low in enumerate(lows[:5]):
        one = (low + sub).astype(np.uint32)
        steps += [(f"one voxel of {k}", one[3:4], 6), (f"the rest of {k}", one, 6),
                  (f"all but one of {k}", one[1:], 0), (f"none of {k}", one, 0)]
    steps += [("filled again", all_of, 7), ("cleared again", all_of, 0)]
    for label, xyz, v in steps:
        apply(w, grid, xyz, np.full(len(xyz), v, np.uint32))
        equals_fresh_world(ctx, layout, w, grid, f"{n}^3 {label}")
    w.close()


@pytest.mark.parametrize("layout,n", [("reference", 64), ("reference", 256), ("dense", 256),
                                      ("dense", 512), ("dense", 1024)])
def test_layer_by_layer(ctx, layout, n):
    """Edits that change a few of the map's layers along z (8 voxels each, 128
    of them at 1024^3): at both ends, on either side of the 64th, at a layer's
    faces, where a voxel is near cells of two; one layer and several at once;
    placed and taken away in another order."""
    rng = np.random.default_rng([n, 8])
    grid = np.zeros((n, n, n), np.uint8)
    grid[n // 4:n // 4 + 9, n // 3:n // 3 + 5, n // 2:n // 2 + 30] = 4
    w = fresh(ctx, layout, grid)
    at = sorted({0, 5, 7, 8, 10, n // 2 - 2, n // 2 - 1, n // 2, n // 2 + 4, n - 9, n - 8, n - 1})
    put = []
    for k, z in enumerate(at):
        xyz = np.stack([rng.integers(0, n, 3), rng.integers(0, n, 3), np.full(3, z)], 1)
        put.append(xyz.astype(np.uint32))
        if k % 3 == 2 or k == len(at) - 1:  # the last few in one call
            apply(w, grid, np.vstack(put[k - k % 3:]), np.full(3 * (k % 3 + 1), 5, np.uint32))
            equals_fresh_world(ctx, layout, w, grid, f"{n}^3 up to layer {z // 8}")
    for k in rng.permutation(len(at)):
        apply(w, grid, put[k], np.zeros(3, np.uint32))
        if k % 3 == 0:
            equals_fresh_world(ctx, layout, w, grid, f"{n}^3 without {at[k]}")
    w.close()
