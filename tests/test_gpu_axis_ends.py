"""Axes whose first or last edge shares a cell of the key table with keys that are uncertain anyway:
spherical axes that end between a right angle and pi (nearly antipodal keys above), axes whose first
edge is -Inf (nearly coincident keys below the second).  Results against the oracle, and the share of
pairs left to the re-bin against what the edges' own intervals hold."""
import numpy as np
import pytest

import _oracle
from test_gpu_parity import MAG, TOL, check, field, gpu_hist

pytestmark = pytest.mark.gpu

SPHERE = [np.geomspace(1e-3, 1.6, 21), np.geomspace(1e-3, 2.0, 21), np.geomspace(1e-2, 2.2, 21),
          np.geomspace(1e-3, 2.4, 33), np.geomspace(1e-3, 2.8, 65), np.geomspace(1e-3, 3.05, 33),
          np.array([0.5, 1.0, 2.0]), np.array([0.0, 2.5]), np.array([-1.0, 0.7, 3.0])]
FLAT = [np.array([-np.inf, 0.5, np.inf]), np.array([-np.inf, 0.25, 0.5, 1.0]), np.array([-np.inf, 1.0, 1.1]),
        np.append(np.insert(np.geomspace(0.125, 1.0, 13), 0, -np.inf), np.inf)]


@pytest.mark.parametrize("geometry,k", [("deg", k) for k in range(len(SPHERE))] + [("flat", k) for k in range(len(FLAT))])
def test_uncertain_share(ctx, geometry, k):
    edges = (SPHERE if geometry == "deg" else FLAT)[k]
    x, u, _ = field(geometry, 2, 2000, 11 + k)
    os_, oc, oa, og = _oracle.hist(x, u, edges, op=(0, 2, 0), geometry=geometry, nthreads=4, with_mag=True)
    for prec in ("fp64", "mixed"):
        gs, gc = gpu_hist(ctx, x, u, edges, (0, 2, 0), geometry=geometry, prec=prec)
        check(gs, gc, os_, oc, oa, TOL[prec], f"{geometry} axis {k} {prec}", og=og, mag=MAG[prec])
        if prec == "mixed":
            # an edge's interval is 2^-19 of its key wide (pairs are spread over the keys: ten times that
            # for the densest), the nearly coincident and antipodal keys hold 2^-22 of all pairs
            st = ctx.stats()
            assert st["rebinned"] <= (10 * 2.0 ** -19 * len(edges) + 2.0 ** -20) * st["pairs"] + 8


def test_thousands_of_bins_near_pi(ctx):
    # 7800 bins between 3.04 rad and nearly pi: the histogram leaves room for the plain key table only
    # (7800 x 20 bytes and a table of 10 KB are more than a workgroup's 160 KB)
    edges = np.linspace(np.pi - 0.1, np.pi - 0.0012, 7801)
    x, u, _ = field("deg", 2, 1500, 5)
    os_, oc, oa, og = _oracle.hist(x, u, edges, op=(0, 2, 0), geometry="deg", nthreads=4, with_mag=True)
    assert oc.sum() > 500
    gs, gc = gpu_hist(ctx, x, u, edges, (0, 2, 0), geometry="deg", prec="fp64")
    check(gs, gc, os_, oc, oa, TOL["fp64"], "bins near pi", og=og, mag=MAG["fp64"])
