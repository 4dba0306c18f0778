"""The list build's candidate test by 16-bit coordinates, emulated on the CPU (no GPU).

The reorder pass stores floor(x kFixedH / h) modulo 65536 of each coordinate (8 h, with
kFixedH steps per h); the list build takes 16-bit differences, which wrap, and
w = dx^2 + dy^2 + dz^2 - kFixedH^2 + kFixedBand in 32 bits.  Negative is a neighbour,
from 2 kFixedBand on is none, and what lies between goes to the FP64 test that the
reference's list follows (neighbors.c:248-290).  Searched cells lie within 2 h.

Checked for several h and positions up to 100 m, with the kernels' own constants:
* a decision without the FP64 test never differs from it: pairs near h, pairs anywhere
  within 2 h per axis, pairs on both sides of every wrap;
* w fits 31 bits, and the rounding stays below kFixedBand;
* a coordinate that is not a number is beyond h of all that share its cells (the first
  two), on one, two or three axes;
* with a band of half the width the same pairs are misclassified, so the check can fail."""
import os
import re

import numpy as np
import pytest

F32 = np.float32
HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sphpc_amd",
                      "csrc", "sph_internal.h")


def constants():
    text = open(HEADER).read()
    h, band = re.search(r"kFixedH = (\d+), kFixedBand = (\d+);", text).groups()
    num, den = re.search(r"kFixedNaN = (\d+) \* kFixedH / (\d+);", text).groups()
    return int(h), int(band), int(num) * int(h) // int(den)


H, BAND, NAN = constants()
RADII = [2.0 * float(F32(s)) for s in (0.0025, 0.008, 0.01, 0.02, 0.03)]


def fixed16(x, h):
    """The reorder pass's coordinate of FP32 positions, as int64."""
    t = x.astype(np.float64) * (H / h)
    with np.errstate(invalid="ignore"):
        v = np.where(np.isnan(x), 0.0, t - 65536.0 * np.floor(t * (1.0 / 65536.0)))
    return np.where(np.isnan(x), NAN, v.astype(np.int64) & 0xFFFF)


def fixed_w(p, q, h, band=BAND):
    d = (fixed16(p, h) - fixed16(q, h) + 32768) % 65536 - 32768  # int16 subtraction
    w = (d * d).sum(1) + (band - H * H)
    assert np.all(np.abs(w) < 1 << 31) and np.all((d * d).sum(1) < 1 << 31)
    return w


def fp64_inside(p, q, h):
    d = p.astype(np.float64) - q.astype(np.float64)
    return d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2] < h * h


def wrong(p, q, h, band=BAND):
    """Decisions taken without the FP64 test that differ from it."""
    w, inside = fixed_w(p, q, h, band), fp64_inside(p, q, h)
    return int(np.sum((w < 0) & ~inside) + np.sum((w >= 2 * band) & inside))


def near(h, n, spread, extent, seed):
    rng = np.random.default_rng(seed)
    p = rng.uniform(0.0, extent, (n, 3)).astype(F32)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    r = h * (1.0 + rng.uniform(-spread, spread, n))
    return p, (p.astype(np.float64) + d * r[:, None]).astype(F32)


@pytest.mark.parametrize("extent", [0.5, 6.0, 100.0])
@pytest.mark.parametrize("h", RADII)
def test_decisions_of_pairs_near_the_radius(h, extent):
    for spread in (1e-6, 1e-4, 2e-3):
        p, q = near(h, 40000, spread, extent, int(h * 1e5))
        assert wrong(p, q, h) == 0
    # some are decided at once on either side, and near h all are left to the FP64 test
    w = fixed_w(p, q, h)
    assert np.any(w < 0) and np.any(w >= 2 * BAND)
    r2 = ((p.astype(np.float64) - q) ** 2).sum(1) * (H / h) ** 2
    assert np.max(np.abs(w - BAND + H * H - r2)) < BAND


@pytest.mark.parametrize("h", RADII)
def test_decisions_of_any_pair_of_searched_cells(h):
    """Up to 2 h on each axis, with the positions around the wraps of 8 h."""
    rng = np.random.default_rng(3)
    n = 200000
    base = rng.integers(0, 12, (n, 3)) * 8.0 * h + rng.uniform(-2.0, 2.0, (n, 3)) * h
    p = np.maximum(base, 0.0).astype(F32)
    q = np.maximum(p + rng.uniform(-2.0, 2.0, (n, 3)) * h, 0.0).astype(F32)
    q[: n // 4] = p[: n // 4]
    axis = rng.integers(0, 3, n // 4)
    q[np.arange(n // 4), axis] += (rng.choice([-2.0, -1.0, 0.0, 1.0, 2.0], n // 4) * h).astype(F32)
    assert wrong(p, q, h) == 0
    d = np.floor(p.astype(np.float64) / (8.0 * h)) != np.floor(q.astype(np.float64) / (8.0 * h))
    assert np.sum(d.any(1)) > n // 10  # pairs with a wrap between them


@pytest.mark.parametrize("axes", [(0,), (1, 2), (0, 1, 2)])
@pytest.mark.parametrize("h", RADII)
def test_not_a_number_has_no_neighbours(h, axes):
    """Its cell on such an axis is the first: the others there lie in the first two."""
    rng = np.random.default_rng(4)
    n = 20000
    p = rng.uniform(0.0, 2.0 * h, (n, 3)).astype(F32)
    p[0], p[1] = 0.0, np.nextafter(F32(2.0 * h), F32(0.0))
    q = p.copy()
    q[:, list(axes)] = np.nan
    assert np.all(fixed_w(p, q, h) >= 2 * BAND) and np.all(fixed_w(q, p, h) >= 2 * BAND)


def test_a_narrower_band_misclassifies():
    h = RADII[2]
    p, q = near(h, 400000, 2e-3, 6.0, 8)
    assert wrong(p, q, h) == 0 and wrong(p, q, h, BAND // 2) > 0
