"""The smallest maps on the GPU vs the oracle: the empty-space iteration takes
up to 6 steps at once and tests the grid's edge once per iteration, by the top
bit of each coordinate, which needs at least 12 blocks a side.  Maps of 8^3
(one chunk; literal loop), 16^3 and 24^3 (not a power of two; literal loop) in
the reference layout, 16^3 and 32^3 dense; a few blocks in the corners and at
random, so that most rays cross the whole map and leave it; cameras in every
octant, on exact diagonals (two and three axes tie at every step), with and
without stored step counts."""
import numpy as np
import pytest

import oracle_ffi as O
import vt
from brickmap_util import embedding_a
from test_gpu_parity import compare, gpu_render, poison
from vt import scenes as S

pytestmark = pytest.mark.gpu

W, H, CAP = 33, 17, 200


def grid_of(n, seed):
    rng = np.random.default_rng([n, seed])
    g = np.zeros((n, n, n), np.uint8)
    for z, y, x in rng.integers(0, n, (3, 3)):
        g[z, y, x] = rng.integers(1, 9)
    for corner in rng.integers(0, 2, (2, 3)) * (n - 1):
        g[tuple(corner)] = rng.integers(1, 9)
    return g


def cameras(n, rng):
    out = []
    for k in range(8):
        sg = np.array([(k & 1), (k >> 1) & 1, (k >> 2) & 1]) * 2 - 1
        c = np.full(3, n / 2.0)
        out.append((c - sg * n, c))                       # an exact diagonal
        out.append((c - sg * n * rng.uniform(0.3, 1.5, 3), rng.uniform(0, n, 3)))
    return out


@pytest.mark.parametrize("n", [8, 16, 24])
def test_reference_layout(ctx, n):
    rng = np.random.default_rng(n)
    for seed in range(2):
        layout = embedding_a(grid_of(n, seed), S.palette())
        w, ow = vt.World.brickmap(ctx, *layout), O.BrickmapWorld(*layout)
        for k, (eye, tgt) in enumerate(cameras(n, rng)):
            cam = vt.look_at(eye, tgt, 60.0)
            sun = (S.SUN, (-0.4, 0.4, -0.4))[k & 1]
            o = O.render(ow, cam, W, H, CAP, CAP, sun)
            for steps in (False, True):
                f = poison(vt.Frame.alloc(W, H, steps=steps))
                vt.render(ctx, w, cam, f, vt.params(W, H, CAP, CAP, sun))
                label = f"{n}^3 world {seed} camera {k} steps {steps}"
                assert np.array_equal(f.hits.cpu().numpy().view(np.uint32), o["hits"]), label
                if steps:
                    assert np.array_equal(f.steps.cpu().numpy().view(np.uint32), o["steps"]), label
        w.close()


@pytest.mark.parametrize("n", [16, 32])
def test_dense(ctx, n):
    rng = np.random.default_rng(n + 1)
    grid = grid_of(n, 5)
    w, ow = vt.World.dense(ctx, grid, S.palette()), O.DenseWorld(grid, S.palette())
    for k, (eye, tgt) in enumerate(cameras(n, rng)):
        cam = vt.look_at(eye, tgt, 60.0)
        sun = (S.SUN, (0.4, -0.4, -0.4))[k & 1]
        compare(gpu_render(ctx, w, cam, W, H, CAP, CAP, sun=sun),
                O.render(ow, cam, W, H, CAP, CAP, sun), label=f"{n}^3 camera {k}")
    w.close()
