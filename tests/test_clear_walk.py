"""The bounds the clearance map's exactness rests on (CPU, binary32).

A stretch that the map shows clear is walked without lookups and without
tracking the block: only the sum T of the crossing times is kept.  Two things
must hold for every state of the walk, for at most 3 x 1024 steps:

* the block follows from T: axis i has crossed round(((within0 - within) +
  d T) / 8) boundaries (negative axes: divided by -8 x 0.999), so the value
  before rounding stays well within 0.5 of the true count;
* the position stays near the line p0 + d T / 8: within 0.001 block per
  crossing of a negative axis (the 0.999 re-anchor) plus rounding, and the
  block a lookup probes (the next one on a positive axis whose within reached
  8) touches the position -- less than the 2 blocks by which cells are widened;

and the walk has crossed at least (|dx| + |dy| + |dz|) T / 8 - 3 boundaries,
which decides whether the step cap comes before a near cell.  The recurrence
is the traversal's, operation by operation in float32, vectorised over rays:
random ones, ones with zero components (the 0.001 substitution), shallow ones,
corner-to-corner ones of mixed signs, exact diagonals from lattice points.
"""
import numpy as np
import pytest

from test_reach_margin import rays

F = np.float32


def starts(dim, seed, count):
    rng = np.random.default_rng([dim, seed])
    out = rays(dim, rng, count)
    for k in range(count // 8):  # lattice starts on exact diagonals: ties every step
        sg = rng.choice([-1.0, 1.0], 3)
        e = np.where(sg > 0, rng.integers(0, dim // 4, 3), rng.integers(3 * dim // 4, dim, 3))
        out.append((e.astype(F), (sg / np.sqrt(3.0)).astype(F)))
    e = np.stack([a for a, _ in out])
    d = np.stack([b for _, b in out])
    return e, np.where(d == 0, F(0.001), d).astype(F)


@pytest.mark.parametrize("dim", [32, 128, 512, 1024])
def test_line_bounds(dim):
    e, d = starts(dim, 0, 600)
    inv = (F(1) / d).astype(F)
    pos = d > 0
    P = np.where(pos, F(8), F(0)).astype(F)
    A = np.where(pos, F(0), F(8) * F(0.999)).astype(F)
    g8 = np.trunc(e * F(8)).astype(np.int64)
    w = ((e * F(8)).astype(F) - g8.astype(F)).astype(F) + (g8 & 7).astype(F)
    G = g8 >> 3
    w0, G0 = w.copy(), G.copy()
    p0 = G0 + w0.astype(np.float64) / 8
    d64 = d.astype(np.float64)
    k = np.where(pos, F(0.125), F(-1.0) / (F(8) * F(0.999))).astype(F)
    T = np.zeros(len(e), F)
    live = np.all((G >= 0) & (G < dim), axis=1)
    worst = {"round": 0.0, "line": 0.0, "probe": 0.0, "steps": 0.0}
    rows = np.arange(len(e))
    for step in range(1, 3 * dim + 8):
        t = ((P - w) * inv).astype(F)
        xy, xz, yz = t[:, 0] < t[:, 1], t[:, 0] < t[:, 2], t[:, 1] < t[:, 2]
        m = np.where(xy & xz, 0, np.where(~xy & yz, 1, 2))
        tm = t.min(axis=1)
        nw = (w + (d * tm[:, None]).astype(F)).astype(F)
        nw[rows, m] = A[rows, m]
        w = np.where(live[:, None], nw, w)
        G[rows, m] += np.where(live, np.where(pos[rows, m], 1, -1), 0)
        T = np.where(live, (T + tm).astype(F), T)
        live &= np.all((G >= 0) & (G < dim), axis=1)
        if not live.any():
            break
        n = np.abs(G - G0)
        x = (((w0 - w).astype(F) + (d * T[:, None]).astype(F)).astype(F) * k).astype(F)
        worst["round"] = max(worst["round"], float(np.abs(x - n)[live].max()))
        assert np.array_equal(np.rint(x)[live].astype(np.int64), n[live])
        line = p0 + d64 * T[:, None].astype(np.float64) / 8
        p = G + w.astype(np.float64) / 8
        worst["line"] = max(worst["line"], float(np.abs(p - line)[live].max()))
        q = G + (w >= 8)  # the probed block; its distance from the line's point
        away = np.maximum(np.maximum(q - line, line - (q + 1)), 0).max(axis=1)
        worst["probe"] = max(worst["probe"], float(away[live].max()))
        short = np.abs(d64).sum(axis=1) * T / 8 - n.sum(axis=1)
        worst["steps"] = max(worst["steps"], float(short[live].max()))
    print(f"[clear] dim {dim}: {worst}")
    assert not live.any(), "every walk leaves the grid"
    assert worst["round"] < 0.25
    assert worst["line"] < dim * 0.001 + 0.2 and worst["probe"] < 1.3
    assert worst["steps"] <= 3.0 + 1e-3
