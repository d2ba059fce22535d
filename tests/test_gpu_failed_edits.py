"""An edit that fails after its first kernels have run: an error that the HIP
runtime still holds from an earlier, unrelated call of the thread is reported
at the edit's first check, when the voxels have been written and the maps have
not been rebuilt.  Whatever voxels the world then holds (vt_world_get_voxels),
its frames must be the oracle's of those voxels -- no ray may skip them by a
map made before -- and so after the same edit again, after another edit and
after a generator run; then the maps and the occupancy levels are current
again (the free-region map and the frames of a fresh world, every traversal).
"""
import ctypes as C

import numpy as np
import pytest

import brickmap_util as BU
import oracle_ffi as O
import vt
from test_gpu_clear import check
from test_gpu_freemap import OFF, ON, SUNS, render_free
from vt import scenes as S

pytestmark = pytest.mark.gpu

N, W, H, CAP = 64, 56, 40, 256


def leave_an_error():
    """An invalid device index: refused by the runtime on the host, which
    keeps the error of the call until it is asked for."""
    vt._native.lib()
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    assert C.CDLL(path).hipSetDevice(9999) != 0


def voxels(w):
    xyz = np.stack(np.meshgrid(*[np.arange(N)] * 3, indexing="ij"), -1).reshape(-1, 3)[:, ::-1]
    return w.get_voxels(xyz.astype(np.uint32)).reshape(N, N, N).astype(np.uint8)


def frames_equal_oracle(ctx, w, layout, label, traversals=(0,)):
    grid = voxels(w)
    ow = O.DenseWorld(grid, S.palette())
    seen = 0
    for k, cam in enumerate((vt.look_at((-20.0, 50.0, -30.0), (32.0, 30.0, 32.0), 70.0),
                             vt.look_at((60.0, 60.0, 60.0), (20.0, 20.0, 20.0), 70.0))):
        o = O.render(ow, cam, W, H, CAP, CAP, SUNS[k])
        seen += int(np.sum(o["hits"][..., 0] != 0xFFFFFFFF))
        for flags in (ON, 0, OFF):
            for t in traversals:
                got = render_free(ctx, w, cam, W, H, CAP, CAP, SUNS[k], flags, gbuffer=False,
                                  traversal=t)
                check(got, o, f"{layout} {label}: camera {k} flags {flags} traversal {t}")
    return grid, seen


def small_world(ctx, layout):
    grid = np.zeros((N, N, N), np.uint8)
    grid[:, 0:3, :] = 3          # a floor, clear space above it
    grid[40:44, 40:44, 40:44] = 5
    if layout == "dense":
        return vt.World.dense(ctx, grid, S.palette())
    w = vt.World.brickmap(ctx, *BU.embedding_a(grid, S.palette()))
    xyz, val = wall()  # half of the wall's chunks have a block, an empty one
    w.set_voxels(xyz[xyz[:, 0] < 32], val[xyz[:, 0] < 32])
    w.set_voxels(xyz[xyz[:, 0] < 32], grid[tuple(xyz[xyz[:, 0] < 32].T[::-1])])
    return w


def wall():
    """A wall in the clear space: of the block at 40..44 and of chunks that
    hold nothing yet."""
    z, y, x = np.mgrid[20:24, 6:46, 16:48]
    xyz = np.stack([x.ravel(), y.ravel(), z.ravel()], 1).astype(np.uint32)
    over = np.stack([v.ravel() for v in np.mgrid[40:48, 44:48, 40:48]], 1).astype(np.uint32)
    return np.vstack([xyz, over]), np.full(len(xyz) + len(over), 6, np.uint32)


@pytest.mark.parametrize("then", ["again", "other"])
@pytest.mark.parametrize("layout", ["dense", "reference"])
def test_edits_after_a_failed_one(ctx, layout, then):
    w = small_world(ctx, layout)
    frames_equal_oracle(ctx, w, layout, "before")
    xyz, val = wall()
    leave_an_error()
    with pytest.raises(vt.VtError):
        w.set_voxels(xyz, val)
    frames_equal_oracle(ctx, w, layout, "after the failed edit")
    if then == "again":
        w.set_voxels(xyz, val)
        assert np.array_equal(w.get_voxels(xyz), val)
    else:  # one voxel that another already makes nonempty: nothing else changes
        w.set_voxels([[5, 1, 5]], [7])
    traversals = (vt.VT_TRAVERSAL_FLAT, vt.VT_TRAVERSAL_BITMASK) if layout == "dense" else (0,)
    grid, seen = frames_equal_oracle(ctx, w, layout, f"then {then}", traversals)
    assert seen > 200
    f = (vt.World.dense(ctx, grid, S.palette()) if layout == "dense"
         else vt.World.brickmap(ctx, *BU.embedding_a(grid, S.palette())))
    a, av = w.read_free_map()
    b, bv = f.read_free_map()
    assert av and bv and np.array_equal(a, b)
    f.close()
    w.close()


def test_generator_run_after_a_failed_edit(ctx):
    """The failed edit's occupancy bytes lie above the layers that the
    generator writes."""
    atlas = BU.embedding_a(np.ones((8, 8, 8), np.uint8), S.palette())[3]
    w, f = (vt.World.empty_brickmap(ctx, 512, atlas) for _ in range(2))
    xyz = np.stack([np.full(60, 100), 440 + np.arange(60), np.full(60, 300)], 1)
    leave_an_error()
    with pytest.raises(vt.VtError):
        w.set_voxels(xyz, np.full(60, 2, np.uint32))
    assert not w.read_brickmap()[0].any()
    for x in (w, f):
        x.procgen(3.0, 4.0)
    a, av = w.read_free_map()
    b, bv = f.read_free_map()
    assert av and bv and np.array_equal(a, b)
    cam = vt.look_at((250.0, 90.0, 250.0), (400.0, 20.0, 300.0), 90.0)
    ra, rb = (render_free(ctx, x, cam, 96, 64, 1024, 512, S.SUN, ON, gbuffer=False)
              for x in (w, f))
    assert np.array_equal(ra["hits"], rb["hits"])
    w.close()
    f.close()
