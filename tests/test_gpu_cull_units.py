"""Work units of culled slices: the device's spatial sort (one and several tiles a workgroup, keys of 8
and of 10 bits an axis, all points in few cells) and the units' rounds (batches of culled and whole slices,
fixed-point flushes) against the same calls that cannot be culled (an infinite last edge adds one bin).

Counts are bit-identical; sums differ by the order of binary64 additions alone (1e-12 of the bin's
sum of magnitudes, here of even orders), fixed-point ones by 2^-22 value-bin widths a pair."""
import numpy as np
import pytest

from sfamd import _native
from test_gpu_parity import gpu_hist

pytestmark = pytest.mark.gpu


def points(n, kind, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(0, 1, (2, n))
    if kind == "cluster":  # all but a few points in one cell of the coarser keys
        x[:, 64:] = 0.3 + 1e-3 * x[:, 64:]
    return x, rng.normal(size=(2, n))


# 2048 keys a tile, 256 workgroups: 530001 points take two tiles each; a reach below 1/32 of the extent
# takes 10-bit keys
@pytest.mark.parametrize("n,kind,reach", [(1024, "even", 0.1), (2049, "even", 0.1), (4097, "even", 0.02),
                                          (6001, "cluster", 2e-4), (530001, "even", 0.004), (530001, "even", 0.05)])
def test_sort_and_units(ctx, n, kind, reach):
    x, u = points(n, kind, n)
    de = np.geomspace(reach / 50, reach, 9)
    s1, c1 = gpu_hist(ctx, x, u, de, (0, 2, 0), prec="mixed")
    culled = ctx.stats()["items"]
    s2, c2 = gpu_hist(ctx, x, u, np.append(de, np.inf), (0, 2, 0), prec="mixed")
    # (1024 points: boxes of 64 leave out less than half of the pairs; one cell: the order is the
    # caller's and the boxes are the cluster's.  Both are evaluated whole.)
    if kind == "even" and n > 2048:
        assert culled < ctx.stats()["items"]
    assert np.array_equal(c1, c2[:-1])
    assert np.all(np.abs(s1 - s2[:-1]) <= 1e-12 * np.abs(s2[:-1]))


def batch(ctx, fields, de, ve, prec):
    keep, probs = [], []
    for x, u in fields:
        x, u, e, v = np.asfortranarray(x), np.asfortranarray(u), np.ascontiguousarray(de), np.ascontiguousarray(ve)
        keep += [x, u, e, v]
        p = _native.SfProblem()
        p.D, p.W, p.N = 2, 2, x.shape[1]
        p.x, p.u = x.ctypes.data, u.ctypes.data
        p.geometry, p.radius = 0, 1.0
        p.op, p.nl, p.nt = 0, 1, 0
        p.n_dist, p.dist_edges = len(e) - 1, e.ctypes.data
        p.n_val, p.val_edges = len(v) - 1, v.ctypes.data
        p.precision, p.count_bits = prec, 64
        probs.append(p)
    nd, nv = len(de) - 1, len(ve) - 1
    s, c = np.zeros(len(fields) * nd * nv), np.zeros(len(fields) * nd * nv, dtype=np.uint64)
    ctx.hist(probs, s, c)
    return s.reshape(len(fields), nv, nd), c.reshape(len(fields), nv, nd)


@pytest.mark.parametrize("prec", ["mixed", "fixed"])
def test_batch_of_culled_and_whole_slices(ctx, prec):
    """Two sizes below the culling threshold, three above, one all within reach (not culled), one slice
    large enough that a round's columns pass the fixed-point flush limit on few workgroups."""
    rng = np.random.default_rng(3)
    fields = [points(n, "even", n) for n in (500, 6001, 3000, 9100, 40000)]
    fields.append((0.01 * rng.uniform(0, 1, (2, 5000)), rng.normal(size=(2, 5000))))
    de, ve = np.geomspace(1e-3, 0.03, 8), np.linspace(-4, 4, 17)
    p = _native.PREC_MIXED if prec == "mixed" else _native.PREC_MIXED_FIXED
    s1, c1 = batch(ctx, fields, de, ve, p)
    ctx.set_tuning(blocks_per_cu=1)
    s3, c3 = batch(ctx, fields, de, ve, p)
    ctx.set_tuning()
    s2, c2 = batch(ctx, fields, np.append(de, np.inf), ve, p)
    width = ve[1] - ve[0]
    for s, c in ((s1, c1), (s3, c3)):
        assert np.array_equal(c, c2[:, :, :-1])
        bound = 1e-12 * 4.0 * c + (2.0 ** -22 * width * c if prec == "fixed" else 0.0)
        assert np.all(np.abs(s - s2[:, :, :-1]) <= bound)
