"""Column groups culled per wave (one-shot calls whose last edge is small against the domain) against
the oracle: sizes at the edges of groups of 32, of 64 of them (one mask), of waves and of row tiles (slices below four row tiles are not culled).

Counts are bit-identical.  Sums: the mixed bound of test_gpu_parity, whose binary32 term is divided
on the sphere by the smallest sine among the counted pairs; fixed-point cells add
1.5 * 2^-23 value-bin widths a pair."""
import numpy as np
import pytest

import _oracle
from test_gpu_parity import MAG, TOL, gpu_hist

pytestmark = pytest.mark.gpu
VE = np.linspace(-3, 3, 31)


@pytest.mark.parametrize("geometry", ["flat2", "flat3", "deg"])
@pytest.mark.parametrize("n", [1055, 2080, 3105, 4101, 6177])
def test_group_edges(ctx, geometry, n):
    rng = np.random.default_rng(n)
    if geometry == "deg":  # scattered points and one dense cluster
        v = rng.normal(size=(3, n))
        v[:, : n // 3] = np.array([0.3, -0.5, 0.8])[:, None] + 0.02 * v[:, : n // 3]
        v /= np.linalg.norm(v, axis=0)
        x = np.degrees(np.stack([np.arctan2(v[1], v[0]), np.arcsin(v[2])]))
        u = rng.normal(size=(2, n))
    else:
        D = 2 if geometry == "flat2" else 3
        x = rng.uniform(0, 1, (D, n))
        x[:, : n // 3] = 0.4 + 0.01 * x[:, : n // 3]
        u = rng.normal(size=(D, n))
    g = "deg" if geometry == "deg" else "flat"
    de = np.geomspace(1e-3, 0.06, 13)
    sin_min = 1e-3 if g == "deg" else 1.0
    for op, ve in [((0, 1, 0), VE), ((0, 2, 0), None), ((0, 0, 3), None)]:
        os_, oc, oa, og = _oracle.hist(x, u, de, op=op, geometry=g, vedges=ve, nthreads=8, with_mag=True)
        for prec in ("mixed", "fixed"):
            if prec == "fixed" and ve is None:
                continue
            gs, gc = gpu_hist(ctx, x, u, de, op, geometry=g, vedges=ve, prec=prec)
            assert np.array_equal(gc, oc), (op, prec)
            bound = TOL["mixed"] * oa + MAG["mixed"] / sin_min * og
            if prec == "fixed":
                bound = bound + 1.5 * 2.0 ** -23 * (ve[1] - ve[0]) * oc
            assert np.all(np.abs(gs - os_) <= bound + 1e-300), (op, prec)
