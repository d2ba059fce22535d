"""Edits and reads through the context's staging, at the sizes where its path
changes: lists of one edit, of exactly the staging's 256 KiB and of more
(device memory of their own), reads over the staging's 16,384 voxels; on both
layouts, with repeated voxels.  After each batch the voxels, the free-region
map (left as it is when no 16^3 region empties or fills) and a frame must be
those of a world made from the edited voxels; and the free-region map of the
largest map (64 regions a side, whole 64-bit rows) its definition's."""
import numpy as np
import pytest

import brickmap_util as BU
import vt
from test_gpu_freemap import boxes_world, expected_free_scan, render_free
from vt import scenes as S

pytestmark = pytest.mark.gpu

# words a list takes: dense 2 an edit + 1 a brick + ..., reference layout 3 + ...
COUNTS = [1, 2, 700, 16384, 16385, 21845, 40000]


def edits(n, count, seed):
    rng = np.random.default_rng([n, count, seed])
    xyz = rng.integers(0, n, (count, 3))
    if count > 100:  # a solid lump (regions fill), some voxels twice
        k = np.arange(count // 2)
        xyz[:len(k)] = np.stack([k % 32, k // 32 % 32, k // 1024 % n], 1)
        xyz[-50:] = xyz[:50]
    return xyz.astype(np.uint32), rng.integers(0, 6, count).astype(np.uint32)


@pytest.mark.parametrize("layout", ["dense", "reference"])
def test_edits_equal_a_fresh_world(ctx, layout):
    n, pal = 128, S.palette()
    grid = boxes_world(n, 3)

    def fresh(g):
        return (vt.World.dense(ctx, g, pal) if layout == "dense"
                else vt.World.brickmap(ctx, *BU.embedding_a(g, pal)))

    w = fresh(grid)
    cam = vt.look_at((-30.0, 100.0, -40.0), (70.0, 40.0, 60.0), 70.0)
    for count in COUNTS:
        xyz, val = edits(n, count, 1)
        w.set_voxels(xyz, val)
        for (x, y, z), v in zip(xyz, val):  # in order: the last write wins
            grid[z, y, x] = v
        got = w.get_voxels(xyz)
        assert np.array_equal(got, grid[xyz[:, 2], xyz[:, 1], xyz[:, 0]]), (layout, count)
        f = fresh(grid)
        a, av = w.read_free_map()
        b, bv = f.read_free_map()
        assert av and bv and np.array_equal(a, b), f"{layout}: free map after {count} edits"
        ra = render_free(ctx, w, cam, 96, 64, 512, 512, S.SUN, flags=0, gbuffer=False)
        rb = render_free(ctx, f, cam, 96, 64, 512, 512, S.SUN, flags=0, gbuffer=False)
        assert np.array_equal(ra["hits"], rb["hits"]), f"{layout}: frame after {count} edits"
        f.close()
    w.close()


def test_large_free_map(ctx):
    n = 1024
    grid = np.zeros((n, n, n), np.uint8)
    rng = np.random.default_rng(9)
    for x, y, z in rng.integers(0, n, (5, 3)):
        grid[z, y, x] = 1
    w = vt.World.dense(ctx, grid, S.palette())
    got, valid = w.read_free_map()
    assert valid and np.array_equal(got, expected_free_scan(grid))
    w.close()
