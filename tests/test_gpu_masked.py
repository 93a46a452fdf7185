"""Fields with masked points (velocities of zero, NaN velocities, NaN positions): every share of them, in
runs and scattered, against the oracle, and the time of such a call against that of the same call without
masked points (their pairs must not be evaluated one by one by the exact sequence)."""
import numpy as np
import pytest

import _oracle
from sfamd import _native
from test_gpu_parity import MAG, TOL, check, field, gpu_hist

pytestmark = pytest.mark.gpu
# value axes with an edge at zero, without one, with one of -0.0, and one that zero lies outside of
AXES = {"even": np.linspace(-4, 4, 25), "odd": np.linspace(-4, 4, 24),
        "negzero": np.concatenate([np.linspace(-4, -1, 5), [-0.0, 0.5, 1.5]]), "above": np.linspace(0.25, 5, 20)}


def mask(x, u, kind, share, run, seed):
    x, u = x.copy(), u.copy()
    n = x.shape[1]
    k = int(round(share * n))
    at = np.arange(n // 3, n // 3 + k) % n if run else np.random.default_rng(seed).permutation(n)[:k]
    if kind == "rest":
        u[:, at] = 0.0
    elif kind == "nan":
        u[seed % u.shape[0], at] = np.nan
    elif kind == "nowhere":
        x[seed % x.shape[0], at] = np.nan if seed % 2 else -np.nan
    return x, u


@pytest.mark.parametrize("prec", ["fp64", "mixed", "fixed"])
@pytest.mark.parametrize("geometry,D", [("flat", 2), ("flat", 3), ("deg", 2), ("deg", 3)])
@pytest.mark.parametrize("kind", ["rest", "nan", "nowhere"])
def test_masked(ctx, geometry, D, kind, prec):
    p = "mixed" if prec == "fixed" else prec
    for k, (share, run) in enumerate([(0.1, False), (0.5, False), (0.4, True), (1.0, False)]):
        x, u, edges = field(geometry, D, 700, 21 + k)
        x, u = mask(x, u, kind, share, run, k)
        cases = [((0, 1, 0), "even"), ((0, 2, 0), "even"), ((0, 1, 0), "odd"), ((0, 1, 0), "negzero"),
                 ((0, 2, 0), "above"), ((1, 0, 0), "even"), ((0, 0, 1), "odd")]
        if prec != "fixed":
            cases += [((0, 2, 0), None), ((2, 0, 0), None), ((0, 0, 3), None), ((1, 0, 0), None)]
        for op, ve in cases:
            ve = None if ve is None else AXES[ve]
            # (fixed-point cells need equal bins; others fall back to the strict ones)
            os_, oc, oa, og = _oracle.hist(x, u, edges, op=op, geometry=geometry, vedges=ve, nthreads=8, with_mag=True)
            gs, gc = gpu_hist(ctx, x, u, edges, op, geometry=geometry, vedges=ve, prec=prec)
            og = np.where(np.isfinite(og), og, 0.0)
            mag = MAG[p] + (16 * 2.0 ** -53 / 1e-4 if prec == "fp64" else 0.0)
            if prec == "fixed":  # 2^-22 value bins a pair
                og = og + oc * (ve[1] - ve[0] if ve is not None else 0.0) * 2.0 ** -22 / mag
            check(gs, gc, os_, oc, oa, TOL[p], f"{geometry} D={D} {kind} {share} {op} {prec}", og=og, mag=mag)


@pytest.mark.parametrize("geometry", ["flat", "deg"])
def test_masked_and_back(ctx, geometry):
    """More columns than the form for such fields runs in one go, masked ones at the start, joint with the
    binary64 kernel: in and out of that form."""
    x, u, edges = field(geometry, 2, 9000, 3)
    u[:, :1500] = 0.0
    u[:, 1500:2000] = np.nan
    os_, oc, oa, og = _oracle.hist(x, u, edges, op=(0, 1, 0), geometry=geometry, vedges=AXES["even"], nthreads=8,
                                   with_mag=True)
    gs, gc = gpu_hist(ctx, x, u, edges, (0, 1, 0), geometry=geometry, vedges=AXES["even"], prec="fp64")
    og = np.where(np.isfinite(og), og, 0.0)
    check(gs, gc, os_, oc, oa, TOL["fp64"], geometry, og=og, mag=16 * 2.0 ** -53 / 1e-4)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("geometry", ["flat", "deg"])
@pytest.mark.parametrize("kind,op,joint", [("rest", (0, 1, 0), True), ("nan", (0, 1, 0), True), ("nan", (0, 2, 0), False),
                                           ("nowhere", (0, 1, 0), True), ("nowhere", (0, 2, 0), False),
                                           ("nowhere", (1, 0, 0), False)])
def test_masked_time(ctx, geometry, kind, op, joint, prec):
    """Kernel time, binary64: at most three times that of the unmasked field (one by one: five to thirteen).
    Binary32: no pair of a NaN position is queued for the re-bin, nor one of two points at rest."""
    x, u, edges = field(geometry, 2, 30000, 5)
    ve = AXES["even"] if joint else None

    def best(x, u):
        t = []
        for _ in range(4):
            gpu_hist(ctx, x, u, edges, op, geometry=geometry, vedges=ve, prec=prec)
            t.append(ctx.stats()["hist_ns"])
        return min(t), ctx.stats()["rebinned"]

    plain, queued = best(x, u)
    for share in (0.3, 1.0):
        xm, um = mask(x, u, kind, share, False, 1)
        t, q = best(xm, um)
        if prec == "fp64":
            assert t <= 3 * plain
        elif kind != "nan":
            assert q <= queued


@pytest.mark.parametrize("geometry,D", [("flat", 2), ("flat", 3), ("deg", 2)])
@pytest.mark.parametrize("ops", [[(1, 0, 0)], [(0, 2, 0), (1, 0, 0)], [(1, 0, 0), (0, 0, 1), (0, 0, 3)], [(0, 0, 0)]])
def test_masked_fused(ctx, geometry, D, ops):
    """Fused outputs of a field with NaN positions of either sign, on axes with closed and open ends, with
    outputs that take the distance and that do not."""
    x, u, edges = field(geometry, D, 500, 41)
    x, u = mask(x, u, "nowhere", 0.2, False, 1)
    x[0, ::7] *= -1.0
    x[0, 3::11] = -np.nan
    axes = [edges, np.concatenate([edges, [np.inf]]), np.concatenate([[-np.inf, 0.0], edges, [np.inf]])]
    for de in axes:
        p = _native.SfProblem()
        xc, uc = np.asfortranarray(x), np.asfortranarray(u)
        p.D, p.W, p.N = uc.shape[0], xc.shape[0], 500
        p.x, p.u = xc.ctypes.data, uc.ctypes.data
        p.geometry, p.radius = _oracle.GEOM[geometry], 1.0
        p.n_dist, p.dist_edges = len(de) - 1, de.ctypes.data
        p.precision, p.count_bits = 1, 64
        outs = []
        for op in ops:
            o = _native.SfOutput()
            o.op, o.nl, o.nt = op
            outs.append(o)
        sums = [np.zeros(len(de) - 1) for _ in ops]
        counts = [np.zeros(len(de) - 1, dtype=np.uint64) for _ in ops]
        ctx.hist_multi([p], outs, sums, counts)
        for k, op in enumerate(ops):
            os_, oc, oa, og = _oracle.hist(x, u, de, op=op, geometry=geometry, nthreads=4, with_mag=True)
            check(sums[k], counts[k], os_, oc, oa, TOL["mixed"], f"{geometry} {op}", og=og, mag=MAG["mixed"])
            gs, gc = gpu_hist(ctx, x, u, de, op, geometry=geometry, prec="mixed")
            check(gs.reshape(-1), gc.reshape(-1), os_, oc, oa, TOL["mixed"], f"{geometry} {op}", og=og, mag=MAG["mixed"])


def test_masked_fused_many_bins(ctx):
    """4500 bins with an open end: 90 KB of LDS for one fused output (eight would need 340 of 160)."""
    x, u, edges = field("flat", 2, 500, 43)
    x, u = mask(x, u, "nowhere", 0.2, False, 1)
    x[0, ::7] *= -1.0
    de = np.append(np.linspace(0.0, edges[-1], 4500), np.inf)
    p = _native.SfProblem()
    xc, uc = np.asfortranarray(x), np.asfortranarray(u)
    p.D, p.W, p.N = uc.shape[0], xc.shape[0], 500
    p.x, p.u = xc.ctypes.data, uc.ctypes.data
    p.geometry, p.radius = _oracle.GEOM["flat"], 1.0
    p.n_dist, p.dist_edges = len(de) - 1, de.ctypes.data
    p.precision, p.count_bits = 1, 64
    o = _native.SfOutput()
    o.op, o.nl, o.nt = 1, 0, 0
    sums, counts = np.zeros(len(de) - 1), np.zeros(len(de) - 1, dtype=np.uint64)
    ctx.hist_multi([p], [o], [sums], [counts])
    os_, oc, oa, og = _oracle.hist(x, u, de, op=(1, 0, 0), geometry="flat", nthreads=4, with_mag=True)
    check(sums, counts, os_, oc, oa, TOL["mixed"], "4500 bins", og=og, mag=MAG["mixed"])


@pytest.mark.parametrize("geometry,D", [("flat", 2), ("flat", 3), ("deg", 2), ("deg", 3)])
@pytest.mark.parametrize("prec", ["fp64", "mixed", "fixed"])
def test_nowhere_open_axes(ctx, geometry, D, prec):
    """NaN positions of either sign on axes with open ends: operators that take the distance and that do not."""
    x, u, edges = field(geometry, D, 500, 61)
    x, u = mask(x, u, "nowhere", 0.2, False, 1)
    x[0, ::7] *= -1.0
    x[0, 3::11] = -np.nan
    p = "mixed" if prec == "fixed" else prec
    for de in (np.append(edges, np.inf), np.concatenate([[-np.inf, 0.0], edges, [np.inf]])):
        for op in ((0, 0, 0), (0, 0, 1), (0, 0, 2), (0, 0, 3), (0, 1, 2), (1, 0, 0), (2, 0, 0), (3, 0, 0), (4, 0, 0), (5, 1, 0),
                   (5, 2, 0), (5, 3, 0)):
            for ve in (None, np.array([-np.inf, 0.0, np.inf]), np.linspace(-4, 4, 24)):
                if prec == "fixed" and ve is None:
                    continue
                os_, oc, oa, og = _oracle.hist(x, u, de, op=op, geometry=geometry, vedges=ve, nthreads=8, with_mag=True)
                gs, gc = gpu_hist(ctx, x, u, de, op, geometry=geometry, vedges=ve, prec=prec)
                og = np.where(np.isfinite(og), og, 0.0)
                mag = MAG[p] + (16 * 2.0 ** -53 / 1e-4 if prec == "fp64" else 0.0)
                if prec == "fixed":  # 2^-22 value bins a pair
                    og = og + oc * 8.0 / 23 * 2.0 ** -22 / mag
                check(gs, gc, os_, oc, oa, TOL[p], f"{geometry} D={D} {op} {prec}", og=og, mag=mag)
