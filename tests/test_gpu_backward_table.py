"""vt_lambert_backward on both sides of the line from which a block sums its
albedo gradients in a table (4096 records a block, 512 blocks at most), vs a
float64 sum over the same records: one record short of the line and at it,
one wave of records, one, and four million; voxels that recur in the whole
image, all in one table, and more voxels than a table has slots; sky between
them; dense and compact albedo; both upstream kinds.

Tolerance: a voxel's n terms are summed in binary32 in some order; the error
is a random walk of n roundings of at most 2^-24 of the sum of their
magnitudes: sqrt(n) 2^-24 < 1.3e-4 for n < 4.2e6, taken as 2e-4 of that sum
(and of the loss and sun gradient's)."""
import numpy as np
import pytest

import vt
from vt import _native as N
from vt import scenes as S

pytestmark = pytest.mark.gpu

DIM, AMBIENT, TOL = 64, 0.2, 2e-4
LINE = 512 * 4095  # npix / 512 + 1 = 4096 records a block from here


@pytest.fixture(scope="module")
def world(ctx):
    rng = np.random.default_rng(2)
    grid = rng.integers(1, 9, (DIM,) * 3).astype(np.uint8)  # voxels to choose from
    grid[rng.random(grid.shape) < 0.2] = 0
    w = vt.World.dense(ctx, grid, S.palette())
    vt.build_compact_index(ctx, w)
    yield w, np.flatnonzero(grid.ravel())
    w.close()


def records(occupied, npix, kind, rng):
    pool = {"few": occupied[:50], "one": occupied[7:8], "all": occupied}[kind]
    rec = np.zeros((npix, 3), np.uint32)
    rec[:, 0] = rng.choice(pool, npix)
    run = rng.random(npix) < 0.6  # runs of equal voxels
    idx = np.maximum.accumulate(np.where(run, 0, np.arange(npix)))
    rec[:, 0] = rec[idx, 0]
    rec[rng.random(npix) < 0.1, 0] = 0xFFFFFFFF
    rec[:, 2] = rng.integers(1, 7, npix) | (rng.integers(0, 2, npix) << 3)
    return rec


def reference(rec, albedo, up, kind):
    """The terms by their definition in binary32, their sums in float64."""
    f = np.float32
    sun = np.array(S.SUN, f)
    ls = np.sqrt(sun[0] * sun[0] + sun[1] * sun[1] + sun[2] * sun[2])
    l = sun / ls
    normals = np.array([[0, 0, 0], [-1, 0, 0], [1, 0, 0], [0, -1, 0], [0, 1, 0], [0, 0, -1],
                        [0, 0, 1]], f)
    hit = rec[:, 0] != 0xFFFFFFFF
    n = normals[rec[:, 2] & 7]
    nd = n[:, 0] * l[0] + n[:, 1] * l[1] + n[:, 2] * l[2]
    vis = np.where((rec[:, 2] >> 3) & 1, f(0), f(1))
    fct = f(AMBIENT) + np.maximum(nd, f(0)) * vis
    voxel = np.where(hit, rec[:, 0], 0).astype(np.int64)
    A = albedo.reshape(-1, 3)[voxel]
    r = np.where(hit[:, None], A * fct[:, None], f(0)) - up[:, :3]
    target = kind == N.VT_UPSTREAM_L2_TARGET
    loss = np.sum(r.astype(np.float64) ** 2) if target else 0.0
    g = np.where(hit[:, None], f(2) * r if target else up[:, :3], f(0))
    ga, mag = np.zeros((DIM ** 3, 3)), np.zeros((DIM ** 3, 3))
    for c in range(3):
        t = (g[:, c] * fct).astype(np.float64)
        ga[:, c] = np.bincount(voxel, t, DIM ** 3)
        mag[:, c] = np.bincount(voxel, np.abs(t), DIM ** 3)
    lit = hit & (nd > 0) & (vis > 0)
    k = np.where(lit, (g[:, 0] * A[:, 0] + g[:, 1] * A[:, 1] + g[:, 2] * A[:, 2]) / ls, f(0))
    terms = (k[:, None] * (n - nd[:, None] * l)).astype(np.float64)
    return ga, mag, terms.sum(0), np.abs(terms).sum(0), loss


@pytest.mark.parametrize("npix,kind,compact,upstream", [
    (1, "one", False, "target"), (64, "few", True, "gradient"), (1025, "all", False, "target"),
    (LINE - 1, "few", False, "target"), (LINE, "few", False, "target"),
    (LINE, "one", True, "gradient"), (LINE + 77, "all", True, "target"),
    (4_194_304, "all", False, "gradient"),
])
def test_against_float64(ctx, world, npix, kind, compact, upstream):
    import torch
    w, occupied = world
    rng = np.random.default_rng([npix, len(kind)])
    rec = records(occupied, npix, kind, rng)
    up = rng.uniform(-1, 1, (npix, 4)).astype(np.float32)
    albedo = rng.uniform(0.05, 1, 3 * DIM ** 3).astype(np.float32)
    ukind = N.VT_UPSTREAM_L2_TARGET if upstream == "target" else N.VT_UPSTREAM_GRADIENT
    table, flags, order = albedo, vt.VT_FLAG_LAMBERT, None
    if compact:
        from test_gpu_lambert import compact_rank
        grid = np.zeros(DIM ** 3, np.uint8)
        grid[occupied] = 1
        ids, rank = compact_rank(grid.reshape((DIM,) * 3))
        table = np.empty((len(ids), 3), np.float32)
        table[rank] = albedo.reshape(-1, 3)[ids]
        table, order, flags = table.ravel(), (ids, rank), flags | vt.VT_FLAG_ALBEDO_COMPACT
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    ga, gs, loss = (torch.zeros(k, device="cuda") for k in (table.size, 3, 1))
    prm = vt.params(1, 1, sun=S.SUN, flags=flags, ambient=AMBIENT, albedo=dev(table))
    vt.lambert_backward(ctx, w, dev(rec.view(np.int32)), prm, dev(up), ukind, ga, gs, loss)
    torch.cuda.synchronize()
    want, mag, wsun, msun, wloss = reference(rec, albedo, up, ukind)
    got = ga.cpu().numpy().reshape(-1, 3)
    if compact:
        full = np.zeros((DIM ** 3, 3), np.float32)
        full[order[0]] = got[order[1]]
        got = full
    assert np.all(np.abs(got - want) <= TOL * mag + 1e-12)
    assert np.all(np.abs(gs.cpu().numpy() - wsun) <= TOL * msun + 1e-12)
    assert abs(float(loss.item()) - wloss) <= TOL * wloss + 1e-12
