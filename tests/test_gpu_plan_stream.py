"""GPU: a plan executed at once on a stream of the caller's (its tables are uploaded on the context's
stream), eagerly and as a graph, against a call on the same data."""
import numpy as np
import pytest

from sfamd import _native
from test_gpu_parity import field

pytestmark = pytest.mark.gpu

# the sums of two launches (of non-negative values) differ by the order of their additions only: fewer
# than 1.2e6 pairs, 2^-53 each
RTOL = 1.2e6 * 2.0 ** -53


def _problems(xs, us, de, ve, geometry, prec):
    out = []
    for x, u in zip(xs, us):
        p = _native.SfProblem()
        p.D, p.W, p.N = u.shape[1], x.shape[1], x.shape[0]
        p.x, p.u = x.data_ptr(), u.data_ptr()
        p.geometry, p.radius, p.op, p.nl, p.nt = geometry, 1.0, 0, 2, 0
        p.n_dist, p.dist_edges = len(de) - 1, de.ctypes.data
        p.n_val, p.val_edges = (0, None) if ve is None else (len(ve) - 1, ve.ctypes.data)
        p.precision, p.count_bits = prec, 64
        out.append(p)
    return out


@pytest.mark.parametrize("geometry", ["flat", "deg"])
@pytest.mark.parametrize("kind", ["fp64", "mixed", "joint", "fused"])
@pytest.mark.parametrize("graph", [False, True])
def test_plan_on_a_stream_of_the_callers(ctx, geometry, kind, graph):
    torch = pytest.importorskip("torch")
    dev = torch.device("cuda:0")
    sizes = [1500, 1, 333]
    xs, us = [], []
    for k, n in enumerate(sizes):
        x, u, _ = field(geometry, 2, 1500, 5 + k)
        x, u = x[:, :n], u[:, :n]
        xs.append(torch.from_numpy(np.ascontiguousarray(x.T)).to(dev))
        us.append(torch.from_numpy(np.ascontiguousarray(u.T)).to(dev))
    de = np.geomspace(1e-3, 1.4, 21)
    ve = np.linspace(0.0, 9.0, 17) if kind == "joint" else None
    prec = 0 if kind == "fp64" else 1
    probs = _problems(xs, us, de, ve, 1 if geometry == "deg" else 0, prec)
    outs = None
    if kind == "fused":
        outs = []
        for nt, nl in ((0, 2), (2, 0)):
            o = _native.SfOutput()
            o.op, o.nl, o.nt = 0, nl, nt
            outs.append(o)
    cells = len(sizes) * (len(de) - 1) * (1 if ve is None else len(ve) - 1)
    bufs = [(torch.zeros(cells, dtype=torch.float64, device=dev), torch.zeros(cells, dtype=torch.int64, device=dev))
            for _ in range(2 if outs else 1)]
    want = [(torch.zeros_like(a), torch.zeros_like(b)) for a, b in bufs]
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    plan = _native.Plan(ctx, probs, outs)
    if outs:
        plan.execute_multi([a.data_ptr() for a, _ in bufs], [b.data_ptr() for _, b in bufs], stream.cuda_stream, graph)
    else:
        plan.execute(bufs[0][0].data_ptr(), bufs[0][1].data_ptr(), stream.cuda_stream, graph)
    assert not plan.sync()
    if outs:
        ctx.hist_multi_device(probs, outs, [a.data_ptr() for a, _ in want], [b.data_ptr() for _, b in want], 0)
    else:
        ctx.hist_device(probs, want[0][0].data_ptr(), want[0][1].data_ptr(), 0)
    torch.cuda.synchronize()
    for (gs, gc), (ws, wc) in zip(bufs, want):
        assert int(wc.sum()) > 0 and torch.equal(gc, wc)
        assert torch.all((gs - ws).abs() <= RTOL * ws.abs())
    plan.close()
