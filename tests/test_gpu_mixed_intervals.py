"""Binary32 kernels: rows past a slice's end, keys in the table's nearly coincident and nearly
antipodal intervals, and joint values too small for a fixed-point step.

Counts are bit-identical to the oracle's.  Sums: the mixed bound of test_gpu_parity, whose binary32
term is divided by the smallest sine that the binary32 pair arithmetic sees (pairs within 2^-10 rad
of antipodal are evaluated in binary64); fixed-point cells add 1.5 * 2^-23 value-bin widths a pair."""
import numpy as np
import pytest

import _oracle
from test_gpu_parity import MAG, TOL, gpu_hist

pytestmark = pytest.mark.gpu
VE = np.linspace(-3, 3, 31)


def _field(geometry, n, seed):
    rng = np.random.default_rng(seed)
    if geometry == "deg":
        v = rng.normal(size=(3, n))
        v /= np.linalg.norm(v, axis=0)
        x = np.degrees(np.stack([np.arctan2(v[1], v[0]), np.arcsin(v[2])]))
        return x, rng.normal(size=(2, n)), np.geomspace(1e-3, np.pi, 17)
    D = 2 if geometry == "flat2" else 3
    return rng.uniform(0, 1, (D, n)), rng.normal(size=(D, n)), np.geomspace(1e-3, 2.0, 17)


def _check(ctx, x, u, de, op, geometry, ve, prec, sin_min=1.0):
    g = "deg" if geometry == "deg" else "flat"
    os_, oc, oa, og = _oracle.hist(x, u, de, op=op, geometry=g, vedges=ve, nthreads=8, with_mag=True)
    gs, gc = gpu_hist(ctx, x, u, de, op, geometry=g, vedges=ve, prec=prec)
    assert np.array_equal(gc, oc)
    bound = TOL["mixed"] * oa + MAG["mixed"] / sin_min * og
    if prec == "fixed":
        bound = bound + 1.5 * 2.0 ** -23 * (ve[1] - ve[0]) * oc
    assert np.all(np.abs(gs - os_) <= bound + 1e-300)


@pytest.mark.parametrize("prec", ["mixed", "fixed"])
@pytest.mark.parametrize("geometry", ["flat2", "flat3", "deg"])
@pytest.mark.parametrize("n", [2, 63, 65, 769, 1025])
def test_sizes(ctx, geometry, n, prec):
    """One pair, and the edges of waves and of row tiles of 768 and 1024."""
    x, u, de = _field(geometry, n, 300 + n)
    _check(ctx, x, u, de, (0, 1, 0), geometry, VE, prec, sin_min=1e-3 if geometry == "deg" else 1.0)
    if prec == "mixed":
        _check(ctx, x, u, de, (0, 2, 0), geometry, None, prec, sin_min=1e-3 if geometry == "deg" else 1.0)


@pytest.mark.parametrize("prec", ["mixed", "fixed"])
def test_antipodal(ctx, prec):
    """Points and their antipodes, moved by 0 .. 1e-2 rad, and coincident points."""
    x, u, _ = _field("deg", 200, 9)
    rng = np.random.default_rng(10)
    far = np.stack([x[0] + 180.0, -x[1]]) + np.degrees(10.0 ** rng.uniform(-7, -2, 200)) * rng.choice([-1, 1], (2, 200))
    far[:, :20] = np.stack([x[0] + 180.0, -x[1]])[:, :20]
    far[1] = np.clip(far[1], -90, 90)
    x = np.concatenate([x, far, x[:, :30]], axis=1)
    u = np.concatenate([u, rng.normal(size=(2, 230))], axis=1)
    de = np.concatenate([[0.0], np.linspace(0.1, 3.1, 9), np.pi - 10.0 ** np.linspace(-2, -6, 9), [np.pi]])
    _check(ctx, x, u, de, (0, 1, 0), "deg", VE, prec, sin_min=2.0 ** -10)
    if prec == "mixed":
        _check(ctx, x, u, de, (0, 2, 0), "deg", None, prec, sin_min=2.0 ** -10)


@pytest.mark.parametrize("geometry", ["flat2", "flat3", "deg"])
@pytest.mark.parametrize("ve", [VE, np.concatenate([[0.0], np.geomspace(1e-6, 20, 40)])])
def test_small_values(ctx, geometry, ve):
    """Velocities over nine decades: most joint values lie below a fixed-point step of their cells
    or in bins of a small width, next to others of full size."""
    x, u, de = _field(geometry, 700, 11)
    u *= 10.0 ** np.random.default_rng(12).uniform(-9, 0, u.shape[1])
    g = "deg" if geometry == "deg" else "flat"
    op = (0, 1, 0) if ve[0] < 0 else (0, 2, 0)
    os_, oc, oa, og = _oracle.hist(x, u, de, op=op, geometry=g, vedges=ve, nthreads=8, with_mag=True)
    for prec in ("mixed", "fixed"):
        gs, gc = gpu_hist(ctx, x, u, de, op, geometry=g, vedges=ve, prec=prec)
        assert np.array_equal(gc, oc)
        bound = TOL["mixed"] * oa + MAG["mixed"] / (1e-3 if geometry == "deg" else 1.0) * og + 1e-300
        if prec == "fixed":
            bound = bound + 1.5 * 2.0 ** -23 * np.diff(ve)[None, :] * oc
        assert np.all(np.abs(gs - os_) <= bound)
