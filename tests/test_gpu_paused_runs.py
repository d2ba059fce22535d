"""Empty-space runs that a wave's last rays leave and take up again (reference
layout with the clearance map), vs the oracle: when three quarters of the rays
that began a run together have come to a block, the others pause.  Sparse
model worlds, so that the rays of one wave meet blocks at very different
depths: a wall close to the eye over part of the image, single models far
off, models without a texel to fall through; every step cap around the
distances; suns of both rules; wide and narrow views, widths that leave waves
part empty."""
import numpy as np
import pytest

import oracle_ffi as O
import vt
from brickmap_util import chunked
from test_gpu_freemap import ON, render_free
from test_gpu_model_walk import layout as model_layout
from vt import scenes as S

pytestmark = pytest.mark.gpu


def layout(n, seed):
    _, _, _, atlas = model_layout(16, 1, 0.0)
    rng = np.random.default_rng([n, seed])
    numbers = np.array([0, 1, 2, 31, 32, 1024, 777, 5000], np.uint32) | np.uint32(1 << 28)
    blocks = np.where(rng.random((n, n, n)) < 0.0015, rng.choice(numbers, (n, n, n)), 0)
    blocks[n // 4, : n // 2, : n // 2] = rng.choice(numbers, (n // 2, n // 2))  # a wall, part way
    blocks[:, 1, :] = rng.choice(numbers, (n, n))                               # a floor
    chunks, pool = chunked(blocks.astype(np.uint32))
    return n, chunks, pool, atlas


@pytest.mark.parametrize("n,w,h", [(32, 40, 24), (64, 61, 33), (128, 96, 40)])
def test_frames_equal_the_oracle(ctx, n, w, h):
    lay = layout(n, 3)
    world, ow = vt.World.brickmap(ctx, *lay), O.BrickmapWorld(*lay)
    rng = np.random.default_rng(n)
    views = [((n * 0.3, n * 0.2, 2.3), (n * 0.55, n * 0.25, n * 1.0), 80.0),
             ((n * 0.9, n * 0.5, n * 0.95), (n * 0.1, n * 0.1, n * 0.1), 50.0)]
    views += [(rng.uniform(0, n, 3), rng.uniform(0, n, 3), 95.0) for _ in range(3)]
    hits = 0
    for k, (eye, tgt, fov) in enumerate(views):
        cam = vt.look_at(eye, tgt, fov)
        sun = (S.SUN, (-0.4, 0.5, -0.3))[k & 1]
        for cap in (7, n // 2, n, 6 * n):
            o = O.render(ow, cam, w, h, cap, cap, sun)
            hits += int(np.sum(o["hits"][..., 0] != 0xFFFFFFFF))
            got = render_free(ctx, world, cam, w, h, cap, cap, sun, ON, gbuffer=False)
            label = f"{n}^3 view {k} cap {cap}"
            assert np.array_equal(got["hits"], o["hits"]), label
            assert np.max(np.abs(got["shaded"] - o["shaded"])) <= 1e-5, label
    assert hits > 1000, hits
    world.close()
