"""The clearance map on the GPU vs the oracle: rays cross the stretches it
shows clear without lookups and end where it shows nothing more ahead, or a
near cell only past the step cap.  Every output but the step counts must be
the oracle's, which takes every step and every lookup.

Sizes from the smallest world with a map (32^3: 4 cells a side) to 1024^3;
boxes, single voxels and a thin slab at the grid's faces and corners, so that
lines graze cells, faces and edges; cameras in and out of the grid in every
octant, on exact diagonals and along the axes; suns of every octant; step caps
below, at and above the distance to the first voxel (the cap decides between a
hit and a miss); the flags ON, OFF and the default rule; both layouts; an edit
that moves a wall into a clear stretch."""
import numpy as np
import pytest

import brickmap_util as BU
import oracle_ffi as O
import vt
from test_gpu_freemap import OFF, ON, SUNS, boxes_world, grazing_cameras, random_cameras, render_free
from vt import scenes as S

pytestmark = pytest.mark.gpu

W, H = 40, 28


def check(got, o, label):
    bad = np.argwhere(np.any(got["hits"] != o["hits"], axis=-1))
    assert not len(bad), f"{label}: {len(bad)} records differ, first at {bad[:3].tolist()}"
    assert np.max(np.abs(got["shaded"] - o["shaded"])) <= 1e-5, label


def world_of(kind, n, seed):
    g = boxes_world(n, seed, n_boxes=3, n_single=6)
    if kind == "faces":  # a slab on one face, bars on two edges, corner voxels
        g[:] = 0
        g[:, 0:2, :] = 3
        g[n - 1, :, n - 1] = 5
        g[:, n - 1, 0] = 6
        for c in ((0, 0, 0), (n - 1, n - 1, n - 1), (0, n - 1, n - 1)):
            g[c] = 7
    return g


def cameras(n, rng):
    c = np.full(3, n / 2.0)
    diag = [vt.look_at(c - s * n, c, 50.0) for s in
            (np.array(v, float) for v in ((1, 1, 1), (-1, 1, -1), (1, -1, 1)))]
    axes = [vt.look_at((-5.0, n / 2 + 0.5, n / 2 + 0.5), (n + 5.0, n / 2 + 0.5, n / 2 + 0.5), 40.0),
            vt.look_at((n / 2, n / 2, n / 2), (n / 2, n / 2, -n), 40.0)]
    return random_cameras(n, rng, 6) + grazing_cameras(n, 2.0, rng, 3) + diag + axes


@pytest.mark.parametrize("kind", ["boxes", "faces"])
@pytest.mark.parametrize("n", [32, 64, 128])
def test_frames_equal_the_oracle(ctx, n, kind):
    rng = np.random.default_rng([n, len(kind)])
    grid, pal = world_of(kind, n, 40 + n), S.palette()
    wd, ow = vt.World.dense(ctx, grid, pal), O.DenseWorld(grid, pal)
    wb = vt.World.brickmap(ctx, *BU.embedding_a(grid, pal))
    for k, cam in enumerate(cameras(n, rng)):
        sun = SUNS[k % len(SUNS)]
        for cap in (3, n // 2, n + k, 4 * n):
            o = O.render(ow, cam, W, H, cap, cap, sun)
            for flags in (ON, 0, OFF):
                label = f"{kind} {n}^3 camera {k} cap {cap} flags {flags}"
                check(render_free(ctx, wd, cam, W, H, cap, cap, sun, flags, gbuffer=False), o,
                      label)
                check(render_free(ctx, wb, cam, W, H, cap, cap, sun, flags, gbuffer=False), o,
                      label + " reference layout")
    wd.close()
    wb.close()


def test_every_cap_around_the_distance(ctx):
    """A wall seen straight on and aslant: for caps one by one around the
    number of steps to it the hit appears at the oracle's cap."""
    n, pal = 64, S.palette()
    grid = np.zeros((n, n, n), np.uint8)
    grid[60, :, :] = 4
    wd, ow = vt.World.dense(ctx, grid, pal), O.DenseWorld(grid, pal)
    for k, cam in enumerate((vt.look_at((32.3, 31.7, -9.0), (32.3, 31.7, 70.0), 8.0),
                             vt.look_at((2.0, 61.0, 1.0), (60.0, 5.0, 62.0), 12.0))):
        full = O.render(ow, cam, 8, 8, 400, 400, S.SUN)
        d = int(np.median(full["steps"] & 0xFFFF))
        seen = set()
        for cap in range(max(1, d - 12), d + 13):
            o = O.render(ow, cam, 8, 8, cap, cap, S.SUN)
            check(render_free(ctx, wd, cam, 8, 8, cap, cap, S.SUN, ON, gbuffer=False), o,
                  f"camera {k} cap {cap}")
            seen.add(float(np.mean(o["hits"][..., 0] != 0xFFFFFFFF)))
        assert min(seen) < 0.5 < max(seen), "the caps straddle the distance"
    wd.close()


@pytest.mark.parametrize("n", [512, 1024])
def test_long_walks(ctx, n):
    """Corner-to-corner stretches (the longest drift and sums) in worlds that
    are empty but for voxels in the corners and a wall moved in by an edit."""
    pal, rng = S.palette(), np.random.default_rng(n)
    grid = np.zeros((n, n, n), np.uint8)
    for c in np.ndindex(2, 2, 2):
        lo = np.array(c) * (n - 6)
        grid[lo[0]:lo[0] + 6, lo[1]:lo[1] + 6, lo[2]:lo[2] + 6] = 1 + (c[0] + 2 * c[1])
    w = vt.World.dense(ctx, grid, pal)
    corners = [np.array(c, float)[::-1] * (n - 6) + 3 for c in np.ndindex(2, 2, 2)]
    cams = [vt.look_at(a + rng.uniform(-30, 30, 3), b, 3.0)
            for a in corners for b in corners if np.abs(a - b).sum() > 1.5 * n]
    for step in range(2):
        ow = O.DenseWorld(grid, pal)
        hits = 0
        for k, cam in enumerate(cams):
            o = O.render(ow, cam, W, H, 4096, 4096, SUNS[k % 4], gbuffer=False)
            check(render_free(ctx, w, cam, W, H, 4096, 4096, SUNS[k % 4], ON, gbuffer=False), o,
                  f"{n}^3 step {step} camera {k}")
            hits += int(np.sum(o["hits"][..., 0] != 0xFFFFFFFF))
        assert hits > 0
        m = n // 2  # a wall across the middle
        z, y, x = np.mgrid[m:m + 1, m - 20:m + 20, m - 20:m + 20]
        xyz = np.stack([x.ravel(), y.ravel(), z.ravel()], 1).astype(np.uint32)
        w.set_voxels(xyz, np.full(len(xyz), 8, np.uint32))
        grid[m:m + 1, m - 20:m + 20, m - 20:m + 20] = 8
    w.close()
