"""Linear axes up to pi on the sphere, whose last edges crowd in chord^2 (the mirrored key table of
binary64 calls, the re-bin of the binary32 ones), against the oracle: bins of every width around where the table is taken
(2 to 300 bins; 300 and a log axis with a tiny first edge keep the plain one), pairs spread evenly, near
coincident and near antipodal.  Counts are bit-identical, sums within the bounds of the parity tests
(whose binary32 term is divided by the smallest sine among the pairs in binary32, 2^-10)."""
import numpy as np
import pytest

import _oracle
import sfamd
from test_gpu_parity import MAG, TOL, gpu_hist

pytestmark = pytest.mark.gpu


def points(n, seed):
    rng = np.random.default_rng(seed)
    v = rng.normal(size=(3, n))
    k = n // 4  # antipodes and neighbours of the first points at separations of 1e-7 to 0.3 rad
    s = 10.0 ** rng.uniform(-7, -0.5, k)
    v /= np.linalg.norm(v, axis=0)
    v[:, k:2 * k] = -v[:, :k] + s * rng.normal(size=(3, k))
    v[:, 2 * k:3 * k] = v[:, :k] + s * rng.normal(size=(3, k))
    v /= np.linalg.norm(v, axis=0)
    return np.degrees(np.stack([np.arctan2(v[1], v[0]), np.arcsin(v[2])])), rng.normal(size=(2, n))


@pytest.mark.parametrize("nd", [2, 7, 20, 63, 100, 300])
def test_linear_axis_to_pi(ctx, nd):
    x, u = points(2500, nd)
    edges = np.linspace(0.0, np.pi, nd + 1)
    ve = np.linspace(-3, 3, 17)
    for op, v in [((0, 2, 0), None), ((0, 0, 3), None), ((0, 1, 0), ve), ((1, 0, 0), ve)]:
        if v is not None and nd > 100:
            continue
        os_, oc, oa, og = _oracle.hist(x, u, edges, op=op, geometry="deg", vedges=v, nthreads=8, with_mag=True)
        for prec in ("fp64", "mixed", "fixed"):
            if prec == "fixed" and v is None:
                continue
            gs, gc = gpu_hist(ctx, x, u, edges, op, geometry="deg", vedges=v, prec=prec)
            assert np.array_equal(gc, oc), (nd, op, prec)
            key = "mixed" if prec == "fixed" else prec
            bound = TOL[key] * oa + MAG[key] * 1024.0 * og
            if prec == "fixed":
                bound = bound + 1.5 * 2.0 ** -23 * (ve[1] - ve[0]) * oc
            assert np.all(np.abs(gs - os_) <= bound + 1e-300), (nd, op, prec)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_rule_axis_and_log_axis(ctx, prec):
    """A LinearBinEdges rule through the public entry, and a log axis whose first edge is tiny."""
    x, u = points(2000, 5)
    b = sfamd.MI355XBackend(0, prec)
    for axis in (sfamd.LinearBinEdges(0.0, np.pi, 81), np.geomspace(1e-7, np.pi, 400)):
        r = sfamd.calculate_structure_function(sfamd.L2SF, x, u, axis, np.uint64, backend=b,
                                               output_type=sfamd.StructureFunctionSumsAndCounts,
                                               distance_metric=sfamd.Haversine(1.0))
        e = sfamd.as_edges(axis)
        f = sfamd.calculate_structure_function(sfamd.L2SF, x, u, axis, np.uint64,
                                               backend=sfamd.MI355XBackend(0, "fp64"),
                                               output_type=sfamd.StructureFunctionSumsAndCounts,
                                               distance_metric=sfamd.Haversine(1.0))
        assert np.array_equal(r.counts, f.counts) and len(e) - 1 == len(r.counts)
        if not isinstance(axis, sfamd.LinearBinEdges):
            _, oc, _ = _oracle.hist(x, u, e, op=(0, 2, 0), geometry="deg", nthreads=8)
            assert np.array_equal(r.counts.astype(np.uint64), oc)
