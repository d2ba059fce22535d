"""The walk inside a model block of the reference layout vs the oracle: texel
masks made from the atlas at creation, voxel steps against them until one is
solid or the ray leaves the block.

Models of every kind: single texels in each corner, planes, checkerboards,
random ones, full ones and ones without a texel (a nonempty block that never
stops a ray); texels whose only nonzero byte is the alpha; model numbers 0,
32767 and ones past 32768 (the atlas wraps) with the solid bit and higher bits
set; neighbouring model blocks, so that walks go from block to block; eyes
outside, between and inside blocks, on exact diagonals and along axes (ties in
the walk); every step cap from 1 to past a block's worth and long ones; stored
step counts and none; the smallest map, one without the fast path (24^3) and
one with a clearance map (32^3)."""
import numpy as np
import pytest

import oracle_ffi as O
import vt
from brickmap_util import chunked, slot_origin
from test_gpu_parity import poison
from vt import scenes as S

pytestmark = pytest.mark.gpu

W, H = 29, 19


def models(rng):
    """(model number, 8^3 texels) pairs."""
    out = []
    for k, (number, kind) in enumerate([(0, "corner"), (1, "random"), (2, "plane"), (31, "checker"),
                                        (32, "empty"), (1024, "alpha"), (32767, "random"),
                                        (777, "full"), (5000, "sparse")]):
        m = np.zeros((8, 8, 8), np.uint32)
        colour = rng.integers(1, 2 ** 32, (8, 8, 8), dtype=np.uint64).astype(np.uint32)
        if kind == "corner":
            for c in ((0, 0, 0), (7, 7, 7), (0, 7, 0)):
                m[c] = 0xFF112233
        elif kind == "plane":
            m[3] = colour[3]
        elif kind == "checker":
            z, y, x = np.indices((8, 8, 8))
            m = np.where((x + y + z) % 2 == 0, colour, 0).astype(np.uint32)
        elif kind == "alpha":
            m[2:5, 2:5, 2:5] = 0xFF000000
        elif kind != "empty":
            density = {"random": 0.15, "full": 1.0, "sparse": 0.02}[kind]
            m = np.where(rng.random((8, 8, 8)) < density, colour, 0).astype(np.uint32)
        out.append((number, m))
    return out


def layout(n, seed, density):
    rng = np.random.default_rng([n, seed])
    atlas = np.zeros((256, 256, 256), np.uint32)
    numbers = []
    for number, m in models(rng):
        ox, oy, oz = slot_origin(number)
        atlas[oz:oz + 8, oy:oy + 8, ox:ox + 8] = m
        numbers += [number | (1 << 28), (number + 32768 * 5) | (1 << 28) | (3 << 29)]
    blocks = np.where(rng.random((n, n, n)) < density,
                      rng.choice(np.array(numbers, np.uint32), (n, n, n)), 0).astype(np.uint32)
    chunks, pool = chunked(blocks)
    return n, chunks, pool, atlas.ravel()


def cameras(n, rng):
    c = np.full(3, n / 2.0)
    out = [vt.look_at(c - s * n, c, 50.0) for s in
           (np.array(v, float) for v in ((1, 1, 1), (-1, 1, 1), (1, -1, -1)))]
    for _ in range(4):
        out.append(vt.look_at(rng.uniform(0, n, 3), rng.uniform(0, n, 3), 90.0))
    out.append(vt.look_at((-3.0, n / 2 + 0.5, n / 2 + 0.25), (n + 3.0, n / 2 + 0.5, n / 2 + 0.25),
                          30.0))
    return out


@pytest.mark.parametrize("n,density", [(8, 0.3), (16, 0.6), (24, 0.2), (32, 0.02)])
def test_frames_equal_the_oracle(ctx, n, density):
    lay = layout(n, 1, density)
    w, ow = vt.World.brickmap(ctx, *lay), O.BrickmapWorld(*lay)
    rng = np.random.default_rng(n)
    hits = 0
    for k, cam in enumerate(cameras(n, rng)):
        sun = (S.SUN, (-0.4, 0.4, -0.4), (0.3, -0.8, 0.4))[k % 3]
        for cap in (1, 2, 3, 5, 9, 14, 30, 400):
            o = O.render(ow, cam, W, H, cap, cap, sun)
            hits += int(np.sum(o["hits"][..., 0] != 0xFFFFFFFF))
            for steps in (False, True):
                f = poison(vt.Frame.alloc(W, H, steps=steps))
                vt.render(ctx, w, cam, f, vt.params(W, H, cap, cap, sun))
                label = f"{n}^3 camera {k} cap {cap} steps {steps}"
                assert np.array_equal(f.hits.cpu().numpy().view(np.uint32), o["hits"]), label
                assert np.max(np.abs(f.shaded.cpu().numpy() - o["shaded"])) <= 1e-5, label
                if steps:
                    assert np.array_equal(f.steps.cpu().numpy().view(np.uint32), o["steps"]), label
    assert hits > 2000, hits
    w.close()
