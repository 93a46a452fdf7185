"""The allocation-free entry near the end of its scratch, against the allocating device entry: spherical
binary64 batches whose second records do not fit beside the rest (run in parts), the 2D single pass (whose
binary64 kernel has no second records), and a batch whose histograms alone do not fit (still refused)."""
import numpy as np
import pytest

from sfamd import _native, synthetic
from test_zz_no_alloc import _problem

pytestmark = pytest.mark.gpu


def _batch(torch, n_slices, n, de, ve, op, prec):
    rng = np.random.default_rng(3)
    x, _ = synthetic.sphere_points(rng, n, n_tracks=2, per_track=64)
    dx = torch.from_numpy(np.ascontiguousarray(x.T)).cuda()
    g = torch.Generator(device="cuda")
    g.manual_seed(4)
    du = torch.randn(n_slices, n, 2, generator=g, device="cuda", dtype=torch.float64)
    probs = [_problem(dx.data_ptr(), du[s].data_ptr(), n, 2, 2, 1, op, de, None, prec) for s in range(n_slices)]
    for p in probs:
        if ve is not None:
            p.n_val, p.val_edges = (len(ve) if op[0] != _native.OP_SINGLE_PASS else len(ve) // 6) - 1, ve.ctypes.data
    return (dx, du), probs


@pytest.mark.parametrize("n_slices,n,op", [(400, 1700, (0, 1, 0)), (5, 100000, (0, 2, 0)),
                                           (1, 180000, (_native.OP_SINGLE_PASS, 0, 0))])
def test_parts(ctx, n_slices, n, op):
    torch = pytest.importorskip("torch")
    if op[0] == _native.OP_SINGLE_PASS:  # six planes a slice
        nd, nv, rows = 8, 6, 6
        ve = np.concatenate([np.linspace(-20, 20, nv + 1)] * 6)
    elif n_slices == 400:
        nd, nv, rows = 64, 96, 1
        ve = np.linspace(-5, 5, nv + 1)
    else:
        nd, nv, rows, ve = 20, 1, 1, None
    de = np.geomspace(1e-3, np.pi, nd + 1)
    keep, probs = _batch(torch, n_slices, n, de, ve, op, 0)
    out = []
    for noalloc in (False, True):
        s = torch.zeros(n_slices, nv * nd * rows, dtype=torch.float64, device="cuda")
        c = torch.zeros(n_slices, nv * nd * rows, dtype=torch.int64, device="cuda")
        torch.cuda.synchronize()
        (ctx.hist_device_noalloc if noalloc else ctx.hist_device)(probs, s.data_ptr(), c.data_ptr(), 0)
        torch.cuda.synchronize()
        out.append((s, c))
        assert ctx.stats()["pairs"] == n_slices * n * (n - 1) // 2 * (6 if op[0] == _native.OP_SINGLE_PASS else 1)
    (s1, c1), (s2, c2) = out
    assert int(c1.sum()) > 0 and torch.equal(c1, c2)
    # the order of the additions differs: a bin's c additions of values around 30 in magnitude at most,
    # each rounded by 2^-53 of a partial sum below 30 c, their errors independent
    assert torch.all((s1 - s2).abs() <= 30.0 * 2.0 ** -53 * c1.double() ** 1.5 + 1e-300)


def test_still_refused(ctx):
    torch = pytest.importorskip("torch")
    de, ve = np.geomspace(1e-3, np.pi, 65), np.linspace(-5, 5, 97)
    keep, probs = _batch(torch, 1600, 64, de, ve, (0, 1, 0), 0)  # 157 MB of histograms
    s = torch.zeros(1600, 64 * 96, dtype=torch.float64, device="cuda")
    c = torch.zeros(1600, 64 * 96, dtype=torch.int64, device="cuda")
    with pytest.raises(Exception, match="allocation-free entry"):
        ctx.hist_device_noalloc(probs, s.data_ptr(), c.data_ptr(), 0)
    torch.cuda.synchronize()
    assert int(c.sum()) == 0
