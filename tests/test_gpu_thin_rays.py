"""Rays whose crossing times are not all ordinary numbers, vs the oracle.  The
empty-space phase picks a step's axis by comparing the crossing times with
the smallest one, which is traceMap's rule only while none of them is NaN; a
direction with a component so small that its reciprocal is huge or infinite
(and 0 x inf possible) has to take the loop with traceMap's own compares.  One
component of every ray is scaled to 1e-20 (still the fast phase), 2^-110 (a
reciprocal past 1e30) or 2^-140 (a denormal: an infinite reciprocal), on each
axis and both signs, from eyes off the block lattice; both layouts; with the
clearance map and without."""
import numpy as np
import pytest

import oracle_ffi as O
import vt
from brickmap_util import embedding_a
from test_gpu_freemap import OFF, ON, boxes_world, render_free
from vt import scenes as S

pytestmark = pytest.mark.gpu

W, H, N = 24, 16, 64


def thin_camera(axis, sign, scale, rng):
    eye = rng.uniform(8.3, N - 8.3, 3)
    tgt = eye + rng.uniform(0.5, 1.0, 3) * rng.choice((-1, 1), 3) * N
    tgt[axis] = eye[axis] + sign * 2 * N
    cam = vt.look_at(eye, tgt, 30.0)
    for k in (0, 4, 8):
        cam.view[k + axis] = cam.view[k + axis] * scale
    return cam


@pytest.mark.parametrize("scale", [1e-20, 2.0 ** -110, 2.0 ** -140])
def test_one_thin_component(ctx, scale):
    rng = np.random.default_rng(7)
    grid, pal = boxes_world(N, 5, n_boxes=3, n_single=40), S.palette()
    wd, ow = vt.World.dense(ctx, grid, pal), O.DenseWorld(grid, pal)
    wb = vt.World.brickmap(ctx, *embedding_a(grid, pal))
    hits = 0
    for axis in range(3):
        for sign in (-1, 1):
            for trial in range(3):
                cam = thin_camera(axis, sign, scale, rng)
                o = O.render(ow, cam, W, H, 200, 200, S.SUN)
                hits += int(np.sum(o["hits"][..., 0] != 0xFFFFFFFF))
                for w, kind in ((wd, "dense"), (wb, "reference")):
                    for flags in (OFF, ON):
                        got = render_free(ctx, w, cam, W, H, 200, 200, S.SUN, flags,
                                          gbuffer=False)
                        label = f"axis {axis} sign {sign} trial {trial} {kind} flags {flags}"
                        assert np.array_equal(got["hits"], o["hits"]), label
    assert hits > 100, hits
    wd.close()
    wb.close()
