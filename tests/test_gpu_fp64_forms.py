"""The binary64 kernel's difference form and its queue of pairs evaluated by the reference's sequence.

Counts are bit-identical to the oracle's.  Sums: two binary64 sequences of a pair agree to a few
2^-53 of the velocities, divided by the sine of the separation on the sphere; the tolerance is
1e-12 of sum |value| plus 16 * 2^-53 / sin of sum ||du||^order (16 roundings of operands no larger
than the velocities, sin the smallest sine among the case's pairs)."""
import time

import numpy as np
import pytest

import _oracle
import sfamd
from sfamd import bins
from test_gpu_parity import gpu_hist
from test_gpu_parity import MAG, TOL, check

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


def _check(ctx, x, u, de, op, geometry, ve, sin_min=1e-3):
    g = "deg" if geometry == "deg" else "flat"
    os_, oc, oa, og = _oracle.hist(x, u, de, op=op, geometry=g, vedges=ve, nthreads=8, with_mag=True)
    gs, gc = gpu_hist(ctx, x, u, de, op, geometry=g, vedges=ve, prec="fp64")
    assert np.array_equal(gc, oc)
    assert np.all(np.abs(gs - os_) <= 1e-12 * oa + 16 * 2.0 ** -53 / sin_min * og + 1e-300)


@pytest.mark.parametrize("geometry", ["flat2", "flat3", "deg"])
@pytest.mark.parametrize("n", [2, 33, 64, 257, 1025])
def test_sizes(ctx, geometry, n):
    """One pair, and the edges of waves, of column groups of 32 and of row tiles of 256 and 1024."""
    x, u, de = _field(geometry, n, 100 + n)
    for op, ve in [((0, 1, 0), VE), ((0, 2, 0), np.concatenate([[0.0], np.geomspace(1e-3, 20, 24)])),
                   ((0, 3, 0), None), ((2, 0, 0), None)]:
        _check(ctx, x, u, de, op, geometry, ve)


@pytest.mark.parametrize("geometry", ["flat2", "flat3", "deg"])
def test_every_pair_queued(ctx, geometry):
    """Equal velocities (every du_L is rounding noise or zero, so every joint pair takes the
    reference's sequence, 1024 of a wave's 32 columns at a time against a queue of 64), and
    coincident points."""
    x, u, de = _field(geometry, 321, 7)
    u[:] = np.array([0.75, -1.5, 0.5])[: u.shape[0], None]
    if geometry == "deg":  # equal components are no equal velocities on the sphere: make them tiny
        u *= 0.0
    de = np.concatenate([[0.0], de])
    x[:, 200:230] = x[:, :30]
    _check(ctx, x, u, de, (0, 1, 0), geometry, VE)
    _check(ctx, x, u, de, (0, 2, 0), geometry, np.linspace(0, 1, 9))
    _check(ctx, x, u, de, (1, 0, 0), geometry, None)


def test_antipodal(ctx):
    """Points and their antipodes, moved by 0 .. 1e-2 rad: the pairs within 2.4e-4 rad of
    antipodal take the reference's sequence, the others the difference form (sin >= 2^-12)."""
    x, u, _ = _field("deg", 200, 9)
    rng = np.random.default_rng(10)
    far = np.stack([x[0] + 180.0, -x[1]]) + np.degrees(10.0 ** rng.uniform(-7, -2, 200)) * rng.choice([-1, 1], (2, 200))
    far[:, :20] = np.stack([x[0] + 180.0, -x[1]])[:, :20]
    far[1] = np.clip(far[1], -90, 90)
    x = np.concatenate([x, far], axis=1)
    u = np.concatenate([u, rng.normal(size=u.shape)], axis=1)
    de = np.concatenate([np.linspace(0.1, 3.1, 9), np.pi - 10.0 ** np.linspace(-2, -6, 9), [np.pi]])
    for op in [(0, 1, 0), (0, 2, 0), (0, 0, 2)]:
        _check(ctx, x, u, de, op, "deg", None, sin_min=2.0 ** -12)
    _check(ctx, x, u, de, (0, 1, 0), "deg", VE, sin_min=2.0 ** -12)


@pytest.mark.parametrize("geometry", ["flat2", "deg"])
def test_non_finite_velocities(ctx, geometry):
    """A NaN and an infinite velocity: same counts and the same pattern of NaN and infinite sums."""
    # the oracle's pairs are summed here: its own (compensated) sums turn a lone infinity into NaN
    x, u, de = _field(geometry, 70, 12)
    u[0, 17] = np.inf
    u[1, 49] = np.nan
    g = "deg" if geometry == "deg" else "flat"
    for op, ve in [((0, 1, 0), None), ((0, 1, 0), VE), ((1, 0, 0), None)]:
        nv = 1 if ve is None else len(ve) - 1
        want = np.zeros((len(de) - 1, nv))
        cnt = np.zeros((len(de) - 1, nv), dtype=np.uint64)
        for i in range(70):
            for j in range(i + 1, 70):
                ok, _, v, db, vb = _oracle.pair(x, u, de, i, j, op=op, geometry=g, vedges=ve)
                vb = 1 if ve is None else vb
                if ok and 1 <= db < len(de) and 1 <= vb <= nv:
                    want[db - 1, vb - 1] += v
                    cnt[db - 1, vb - 1] += 1
        gs, gc = gpu_hist(ctx, x, u, de, op, geometry=g, vedges=ve, prec="fp64")
        gs, gc = gs.reshape(want.shape), gc.reshape(want.shape)
        assert np.array_equal(gc, cnt)
        assert np.array_equal(np.isnan(gs), np.isnan(want)) and np.array_equal(np.isinf(gs), np.isinf(want))


@pytest.mark.parametrize("D", [2, 3])
def test_squared_increment_takes_no_direction(ctx, D):
    # |du|^2 (S2, FullVector{2}) of flat fields forms no du_L: its kernel is not slower than du_L^2's
    rng = np.random.default_rng(D)
    x, u = rng.uniform(size=(D, 30000)), rng.normal(size=(D, 30000))
    edges = np.geomspace(1e-2, 1.9, 49)

    def kernel_ns(op):
        t = []
        for _ in range(5):
            gpu_hist(ctx, x, u, edges, op)
            t.append(ctx.stats()["hist_ns"])
        return min(t)

    square = kernel_ns((0, 2, 0))
    assert kernel_ns((1, 0, 0)) <= square and kernel_ns((5, 2, 0)) <= square
    for op in ((1, 0, 0), (5, 2, 0)):
        os_, oc, oa, og = _oracle.hist(x[:, :3001], u[:, :3001], edges, op=op, geometry="flat", nthreads=4, with_mag=True)
        gs, gc = gpu_hist(ctx, x[:, :3001], u[:, :3001], edges, op)
        check(gs, gc, os_, oc, oa, TOL["fp64"], f"{D}D {op}", og=og, mag=MAG["fp64"])


@pytest.mark.parametrize("geometry", ["flat2", "flat3", "deg"])
def test_crowded_axis(ctx, geometry):
    # thousands of bins in the key table's cells: most pairs' distance bins are uncertain, on linear
    # axes, axes of unequal bins and open ones
    rng = np.random.default_rng(8)
    x, u, _ = _field(geometry, 2500, 8)
    top = np.pi if geometry == "deg" else np.sqrt(x.shape[0])
    geo = "deg" if geometry == "deg" else "flat"
    for de in (np.linspace(0.0, top, 1501), np.sort(rng.uniform(0.2, top, 900)),
               np.concatenate([[-np.inf, 0.0], np.sort(rng.uniform(0.0, top, 700)), [np.inf]])):
        for op in ((0, 2, 0), (0, 3, 0), (0, 0, 1), (1, 0, 0), (2, 0, 0)):
            os_, oc, oa, og = _oracle.hist(x, u, de, op=op, geometry=geo, nthreads=8, with_mag=True)
            gs, gc = gpu_hist(ctx, x, u, de, op, geometry=geo)
            check(gs, gc, os_, oc, oa, TOL["fp64"], f"{geometry} {op}", og=og, mag=16 * 2.0 ** -53 / 1e-4)

    # the linear rule, and the time of a call with 600 bins by it against 60
    be = sfamd.MI355XBackend(0, "fp64")

    def call(x, u, nd):
        kw = dict(distance_metric=sfamd.Haversine(1.0)) if geometry == "deg" else {}
        return sfamd.calculate_structure_function(sfamd.L2SF, x, u, bins.LinearBinEdges(0.0, top, nd + 1), np.uint64,
                                                  backend=be, output_type=sfamd.StructureFunctionSumsAndCounts, **kw)

    _, oc, _ = _oracle.hist(x, u, bins.LinearBinEdges(0.0, top, 1501), op=(0, 2, 0), geometry=geo)
    assert np.array_equal(np.asarray(call(x, u, 1500).counts).astype(np.uint64), oc)
    big = _field(geometry, 60000, 9)

    def seconds(nd):
        t = []
        for _ in range(4):
            t0 = time.perf_counter()
            call(big[0], big[1], nd)
            t.append(time.perf_counter() - t0)
        return min(t)

    assert seconds(600) <= (9.0 if geometry == "deg" else 3.8) * seconds(60)
