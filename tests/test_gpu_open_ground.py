"""Worlds that are mostly ground under an open sky.  Their rays leave the
surface into empty space, so by default they take the clearance map although
most of its cells are near something (solid ground is): a frame must not take
the time of one that walks every ray to the edge of the grid.  And worlds that
edits move across the rule's line, with caps on either side of it: every frame
is the oracle's."""
import numpy as np
import pytest

import brickmap_util as BU
import oracle_ffi as O
import vt
from test_gpu_clear import check
from test_gpu_freemap import OFF, SUNS, render_free
from vt import scenes as S

pytestmark = pytest.mark.gpu


def ground(n, share):
    """Solid up to a wavy surface at about this share of the height."""
    t = np.arange(n) / n * 2 * np.pi
    h = n * share + 2 * np.sin(3 * t)[None, :] + 2 * np.cos(5 * t)[:, None]   # [z, x]
    return np.where(np.arange(n)[None, :, None] < h[:, None, :], 3, 0).astype(np.uint8)


def full_chunks(grid, pal):
    """Embedding A of a large grid (BU.embedding_a goes voxel by voxel)."""
    n, m = grid.shape[0], grid.shape[0] // 8
    b = grid.reshape(m, 8, m, 8, m, 8).transpose(0, 2, 4, 1, 3, 5).reshape(m ** 3, 512)
    some = np.flatnonzero(b.any(1))
    chunks = np.zeros(m ** 3, np.uint32)
    chunks[some] = np.arange(1, len(some) + 1)
    return n, chunks, b[some].astype(np.uint32).ravel(), BU.embedding_a(
        np.zeros((8, 8, 8), np.uint8), pal)[3]


def frame_us(ctx, w, cam, flags):
    import torch
    f = vt.Frame.alloc(1280, 720, schedule=False)
    prm = vt.params(1280, 720, 2048, 2048, S.SUN, flags)
    best = float("inf")
    for _ in range(6):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(8):
            vt.render(ctx, w, cam, f, prm)
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) / 8 * 1e3)
    return best


@pytest.mark.parametrize("share", [0.55, 0.7])
@pytest.mark.parametrize("layout", ["dense", "reference"])
def test_rays_into_the_sky_end(ctx, layout, share):
    n, pal = 512, S.palette()
    grid = ground(n, share)
    w = (vt.World.dense(ctx, grid, pal) if layout == "dense"
         else vt.World.brickmap(ctx, *full_chunks(grid, pal)))
    y = n * share
    cam = vt.look_at((n * 0.2, y + 40.0, n * 0.3), (n * 0.8, y - 10.0, n * 0.7), 70.0)
    by_default, off = frame_us(ctx, w, cam, 0), frame_us(ctx, w, cam, OFF)
    print(f"{layout} {share}: {by_default:.1f} us by default, {off:.1f} with the maps off",
          flush=True)
    assert by_default < 0.75 * off
    w.close()


@pytest.mark.parametrize("layout", ["dense", "reference"])
def test_edits_across_the_line(ctx, layout):
    """Blocks added to every cell of the lower, then of the whole sky, and
    taken away again."""
    n, pal = 64, S.palette()
    grid = ground(n, 0.3)
    w = (vt.World.dense(ctx, grid, pal) if layout == "dense"
         else vt.World.brickmap(ctx, *BU.embedding_a(grid, pal)))
    cams = [vt.look_at((-20.0, 50.0, -30.0), (32.0, 20.0, 32.0), 70.0),
            vt.look_at((40.0, 30.0, 40.0), (10.0, 40.0, 20.0), 80.0)]
    z, y, x = (v.ravel() for v in np.mgrid[4:n:8, 28:n:8, 4:n:8])
    low = y < 46
    steps = [(np.zeros(0, int), 0), (np.flatnonzero(low), 5), (np.flatnonzero(~low), 6),
             (np.flatnonzero(low), 0), (np.flatnonzero(~low), 0)]
    for k, (at, value) in enumerate(steps):
        w.set_voxels(np.stack([x[at], y[at], z[at]], 1), np.full(len(at), value, np.uint32))
        grid[z[at], y[at], x[at]] = value
        ow = O.DenseWorld(grid, pal)
        for c, cam in enumerate(cams):
            for caps in ((192, 48), (512, 192), (1024, 1024)):
                o = O.render(ow, cam, 56, 40, *caps, SUNS[c])
                check(render_free(ctx, w, cam, 56, 40, *caps, SUNS[c], 0, gbuffer=False), o,
                      f"{layout} step {k} camera {c} caps {caps}")
    w.close()
