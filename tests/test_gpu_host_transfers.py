"""Host calls' transfers: inputs and tables below and above the page-locked staging size (1 MiB), slices
that share positions, slices with tables of their own, and the coordinate magnitudes that device calls
reduce on the device (more slices than one launch takes, NaN coordinates among them).

Host and device entries run the same kernels on the same data: counts are equal, and sums differ by
the order of binary64 additions only (at most N^2 / 2 = 5.4e8 of them, 2^-53 each, in all 1e-7 of
sum |value| in the worst case; errors of either sign, so 1e-11 is far from what they reach)."""
import numpy as np
import pytest
import torch

import _oracle
from sfamd import _native
from test_gpu_parity import gpu_hist

pytestmark = pytest.mark.gpu


def _problem(x, u, de, prec, keep, device):
    xc, uc = np.asfortranarray(x), np.asfortranarray(u)
    p = _native.SfProblem()
    p.D, p.W, p.N = uc.shape[0], xc.shape[0], xc.shape[1]
    if device:
        xt, ut = torch.from_numpy(xc.T.copy()).cuda(), torch.from_numpy(uc.T.copy()).cuda()
        p.x, p.u = xt.data_ptr(), ut.data_ptr()
        keep += [xt, ut]
    else:
        p.x, p.u = xc.ctypes.data, uc.ctypes.data
    keep += [xc, uc, de]
    p.geometry, p.radius = 0, 1.0
    p.op, p.nl, p.nt = 0, 2, 0
    p.n_dist, p.dist_edges = len(de) - 1, de.ctypes.data
    p.n_val, p.precision, p.count_bits = 0, prec, 64
    return p


def _both(ctx, fields, edges, prec):
    """(sums, counts) of the host and of the device entry."""
    n, nd = len(fields), len(edges[0]) - 1
    keep = []
    hs, hc = np.zeros(n * nd), np.zeros(n * nd, dtype=np.uint64)
    ctx.hist([_problem(x, u, de, prec, keep, False) for (x, u), de in zip(fields, edges)], hs, hc)
    ds = torch.zeros(n * nd, device="cuda", dtype=torch.float64)
    dc = torch.zeros(n * nd, device="cuda", dtype=torch.int64)
    ctx.hist_device([_problem(x, u, de, prec, keep, True) for (x, u), de in zip(fields, edges)], ds.data_ptr(),
                    dc.data_ptr(), 0)
    torch.cuda.synchronize()
    return hs, hc, ds.cpu().numpy(), dc.cpu().numpy().astype(np.uint64)


@pytest.mark.parametrize("prec", [_native.PREC_FP64, _native.PREC_MIXED])
@pytest.mark.parametrize("n", [1, 2, 1000, 32768, 32769])
def test_sizes(ctx, n, prec):
    """x and u of 32768 points in 2D fill the staging buffer."""
    rng = np.random.default_rng(n)
    x, u = 1e3 * rng.uniform(-1, 1, (2, n)), rng.normal(size=(2, n))
    hs, hc, ds, dc = _both(ctx, [(x, u)], [np.linspace(0.0, 3000.0, 41)], prec)
    assert np.array_equal(hc, dc) and int(hc.sum()) == n * (n - 1) // 2
    assert np.all(np.abs(hs - ds) <= 1e-11 * np.abs(ds))


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_batches(ctx, prec):
    """40 slices of 0 to 300 points: shared positions, edges of their own, magnitudes over 12 decades, a
    NaN coordinate (its pairs are in no bin)."""
    rng = np.random.default_rng(5)
    fields, edges = [], []
    for k in range(40):
        n = int(rng.integers(0, 300))
        if k % 4 == 1 and k > 1:
            x = fields[-1][0]
        else:
            x = 10.0 ** (k % 13 - 6) * rng.uniform(-1, 1, (2, n))
        u = rng.normal(size=x.shape)
        fields.append((x, u))
        edges.append(edges[-1] if k % 3 == 1 else np.geomspace(1e-3, 3.0, 21) * 10.0 ** (k % 13 - 6))
    fields[7][0][:, :1] = np.nan
    hs, hc, ds, dc = _both(ctx, fields, edges, {"fp64": 0, "mixed": 1}[prec])
    assert np.array_equal(hc, dc)
    for k, ((x, u), de) in enumerate(zip(fields, edges)):
        if x.shape[1] < 2:
            continue
        os_, oc = _oracle.hist(x, u, de, op=(0, 2, 0))[:2]
        assert np.array_equal(hc[k * 20:(k + 1) * 20], oc), k
    assert np.all(np.abs(hs - ds) <= 1e-11 * np.abs(ds))
