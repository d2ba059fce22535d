"""The rules by which the kernels replace divisions, restated on the CPU and
compared with the divisions themselves.

* a / x as the rounded product of a with a binary64 reciprocal of x that is
  good to 2^-52: equal to the binary32 quotient for ordinary sizes, at random
  and at the quotients closest to a rounding boundary; pixel coordinates over
  image sizes for the whole range of an axis.
* b / 255 for the 256 integers, by a product and one correction; and that a
  colour byte survives the round trip through rgba8.
* traceEntities' five boxes: the wider box around all of them is met whenever
  the exact test meets one, for origins in and next to grids up to 4096^3 and
  directions over twelve decades."""
from fractions import Fraction

import numpy as np
import pytest

f32, f64 = np.float32, np.float64


def check_quotients(a, x, label):
    want = a / x
    for rel in (0.0, 2.0 ** -52, -(2.0 ** -52)):
        y = (1.0 / x.astype(f64)) * (1.0 + rel)
        got = (a.astype(f64) * y).astype(f32)
        bad = got != want
        assert not bad.any(), (label, rel, a[bad][:3], x[bad][:3])


@pytest.mark.parametrize("lo,hi", [(-2.0, 2.0), (-60.0, 60.0)])
def test_quotient_random(lo, hi):
    rng = np.random.default_rng(3)
    n = 2_000_000
    x = (rng.uniform(1, 2, n) * 2.0 ** rng.uniform(lo, hi, n)).astype(f32)
    a = (rng.uniform(1, 2, n) * 2.0 ** rng.uniform(lo, hi, n)).astype(f32)
    check_quotients(a * rng.choice((-1, 1), n).astype(f32), x, "random")


def test_quotient_next_to_boundaries():
    """For a random divisor X (24 bits) the integers A with (2 K + 1) X = 2^25 A
    + r, |r| small, K of 24 bits: quotients as close to a midpoint as 24-bit
    operands allow."""
    rng = np.random.default_rng(4)
    A, X = [], []
    for x in (rng.integers(1 << 23, 1 << 24, 20000) | 1).tolist():
        inv = pow(x, -1, 1 << 25)
        for r in (1, -1, 3, -3):
            m = (r * inv) % (1 << 25)  # m x = r mod 2^25, m odd
            m += 0 if m >= (1 << 24) else (1 << 25)
            a = (m * x - r) >> 25
            if (1 << 23) <= a < (1 << 24):
                A.append(a)
                X.append(x)
    assert len(A) > 20000
    check_quotients(np.array(A, f32), np.array(X, f32), "boundary")


@pytest.mark.parametrize("size", [1, 2, 3, 7, 33, 255, 640, 999, 1080, 1920, 2560, 4093, 65535])
def test_pixel_coordinates(size):
    p = np.arange(size, dtype=f32)
    got = (p.astype(f64) * (1.0 / f64(size))).astype(f32)
    assert np.array_equal(got, p / f32(size))


def rounded(q):
    """The binary32 number nearest to a fraction (no ties arise here)."""
    c = f32(float(q))
    near = [c, np.nextafter(c, f32(-np.inf)), np.nextafter(c, f32(np.inf))]
    return min(near, key=lambda v: abs(Fraction(float(v)) - q))


def test_over_255():
    r = f32(1.0) / f32(255.0)
    for b in range(256):
        q = f32(b) * r
        e = rounded(Fraction(b) - 255 * Fraction(float(q)))
        got = rounded(Fraction(float(e)) * Fraction(float(r)) + Fraction(float(q)))
        assert got == f32(b) / f32(255.0), b
        again = np.floor(got * f32(255.0) + f32(0.5))
        assert again == b


BOXES = np.array([[256, 21, 256], [251, 21, 259], [253, 21, 256], [251, 21, 256],
                  [257, 21, 261]], f32)


def test_entity_boxes_lie_in_the_wider_box():
    rng = np.random.default_rng(5)
    n = 400_000
    o = rng.uniform(-1, 4096, (n, 3)).astype(f32)
    o[::2] = (BOXES[rng.integers(0, 5, n // 2)] + rng.uniform(-40, 40, (n // 2, 3))).astype(f32)
    o[::8] = np.ceil(o[::8])  # lattice points, as shadow origins are
    target = (BOXES[rng.integers(0, 5, n)] + rng.choice((0.0, 0.5, 1.0), (n, 3))
              + rng.uniform(-1e-3, 1e-3, (n, 3))).astype(f32)
    d = (target - o) * (10.0 ** rng.uniform(-6, 6, (n, 1))).astype(f32)
    d = np.where(np.abs(d) > 1e-18, d, f32(1e-18)).astype(f32)
    hit = np.zeros(n, bool)
    with np.errstate(all="ignore"):
        for b in BOXES:
            t0, t1 = (b - o) / d, (b + f32(1) - o) / d
            hit |= np.min(np.maximum(t0, t1), 1) >= np.max(np.minimum(t0, t1), 1)
        inv = f32(1) / d
        lo = np.array([250.99, 20.99, 255.99], f32)
        hi = np.array([258.01, 22.01, 262.01], f32)
        a, b = (lo - o) * inv, (hi - o) * inv
        may = np.max(np.minimum(a, b), 1) <= np.min(np.maximum(a, b), 1)
    assert 1000 < hit.sum() < n
    assert not (hit & ~may).any()
