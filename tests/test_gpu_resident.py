"""Launches on both sides of the line up to which a frame's waves are all
resident at once (five blocks of 16x16 pixels a compute unit: 1280 blocks on
256): up to it the empty-space phase runs an iteration ahead of its lookups,
past it in place.  A frame of exactly 1280 blocks, one of a block column more
and a ragged small one, vs the oracle: the reference composite with caps of
both iteration lengths and caps below one iteration, suns of either rule
(positive on every axis or not), and Lambert frames, whose shading is compared
with the records' own shading pass."""
import numpy as np
import pytest

import oracle_ffi as O
import vt
from test_gpu_freemap import OFF, boxes_world, render_free
from vt import scenes as S

pytestmark = pytest.mark.gpu

N = 64
SIZES = [(640, 512), (656, 512), (37, 21)]


@pytest.fixture(scope="module")
def scene():
    return boxes_world(N, 11, n_boxes=4, n_single=60), S.palette()


def cams():
    inside = vt.look_at((8.3, 40.2, 9.7), (50.0, 20.0, 47.0), 80.0)
    outside = vt.look_at((-30.0, 70.0, 95.5), (32.0, 25.0, 30.0), 55.0)
    return inside, outside


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("cap", [4, 60, 700])
def test_both_sides_equal_the_oracle(ctx, scene, size, cap):
    w, h = size
    world, ow = vt.World.dense(ctx, *scene), O.DenseWorld(*scene)
    for k, cam in enumerate(cams()):
        sun = (S.SUN, (-0.5, 0.7, -0.2))[k]
        o = O.render(ow, cam, w, h, cap, cap, sun)
        got = render_free(ctx, world, cam, w, h, cap, cap, sun, OFF, gbuffer=False)
        label = f"{w}x{h} cap {cap} camera {k}"
        assert np.array_equal(got["hits"], o["hits"]), label
        assert np.max(np.abs(got["shaded"] - o["shaded"])) <= 1e-5, label
    world.close()


@pytest.mark.parametrize("size", SIZES)
def test_lambert_frames(ctx, scene, size):
    import torch
    w, h = size
    world, ow = vt.World.dense(ctx, *scene), O.DenseWorld(*scene)
    albedo = torch.rand(3 * N ** 3, generator=torch.Generator().manual_seed(1)).cuda()
    for k, cam in enumerate(cams()):
        prm = vt.params(w, h, 700, 700, S.SUN, OFF | vt.VT_FLAG_LAMBERT, 0, 0.25, albedo)
        f = vt.render(ctx, world, cam, vt.Frame.alloc(w, h), prm)
        o = O.render(ow, cam, w, h, 700, 700, S.SUN)
        assert np.array_equal(f.hits.cpu().numpy().view(np.uint32), o["hits"]), (size, k)
        out = torch.empty_like(f.shaded)
        vt.lambert_shade(ctx, world, f.hits, prm, out)
        assert torch.equal(f.shaded, out), (size, k)
    world.close()
