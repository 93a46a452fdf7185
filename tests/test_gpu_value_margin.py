"""Binary32 joint calls over uniform value edges: the share of pairs left to the re-bin, against the pairs
whose exact value lies within the margin that the binary32 value and its bin number need, and the time that
their queue takes where it is large (value edges at zero, distance bins that share cells of the key table)."""
import numpy as np
import pytest

from sfamd import synthetic
from test_gpu_parity import gpu_hist

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nv,half", [(512, 4.0), (1024, 4.0), (256, 2.0)])
def test_share_near_uniform_value_edges(ctx, nv, half):
    rng = np.random.default_rng(nv)
    n = 1500
    x = rng.uniform(0, 1, (2, n))
    u = rng.normal(size=(2, n))
    ve = np.linspace(-half, half, nv + 1)  # an edge at zero, where the values crowd; exact in binary32
    gpu_hist(ctx, x, u, np.array([1e-6, 2.0]), (0, 1, 0), vedges=ve, prec="mixed")
    st = ctx.stats()
    i, j = np.triu_indices(n, 1)
    dx, du = x[:, j] - x[:, i], u[:, j] - u[:, i]
    w = 2 * half / nv
    t = ((du * dx).sum(0) / np.sqrt((dx * dx).sum(0)) + half) / w
    unit = 2.0 ** -24
    norm = np.sqrt((u * u).sum(0))
    value = 16 * unit * (norm[i] + norm[j]) / w  # the value's bound, in bins
    edges = 4 * unit * (1 + half / w) + 4 * unit * nv + 1e-6  # v0, 1 / w and -v0 / w in binary32
    bins = 4 * unit * (nv + 2)  # the bin number and its two offsets
    want = np.count_nonzero(np.abs(t - np.rint(t)) <= value + edges + bins)
    assert st["rebinned"] <= 1.03 * want + 10


@pytest.mark.parametrize("op,nd,nv,half,prec", [((0, 0, 3), 64, 64, 4.0, "mixed"), ((0, 3, 0), 64, 64, 0.5, "mixed"),
                                                ((0, 0, 3), 48, 64, 4.0, "fixed"), ((0, 2, 1), 48, 64, 0.5, "fixed")])
def test_third_order_queue(ctx, op, nd, nv, half, prec):
    # 2 to 5 % of the pairs are queued: their reservations in the global queue must not bound the kernel
    x, u, de, _ = synthetic.config4(N=40000)
    m = 2.0 * float(np.sum(np.var(u, axis=1)))
    de = np.geomspace(de[0], np.pi, nd + 1)

    def kernel_us(op, half):
        t = []
        for _ in range(4):
            gpu_hist(ctx, x, u, de, op, geometry="deg", vedges=np.linspace(-half, half, nv + 1), prec=prec)
            st = ctx.stats()
            t.append(st["hist_ns"])
        return min(t), st["rebinned"] / st["pairs"]

    plain, few = kernel_us((0, 0, 1), 2.0 * m ** 0.5)
    cube, many = kernel_us(op, half * m ** 1.5)
    assert few < 0.005 and many > 0.01
    assert cube <= 1.7 * plain


def test_crowded_axis_keeps_its_threads(ctx):
    # a linear axis whose largest keys share cells, on points that have few such distances: room for their
    # pairs in the queue must not cost most of the threads
    rng = np.random.default_rng(4)
    n = 18000
    x = np.cumsum(rng.normal(scale=0.002, size=(2, n)), axis=1) % 1.0
    u = rng.normal(size=(2, n))

    def kernel_ns(nd):
        t = []
        for _ in range(6):
            gpu_hist(ctx, x, u, np.linspace(0.0, np.sqrt(2), nd + 1), (0, 2, 0), prec="mixed")
            t.append(ctx.stats()["hist_ns"])
        return min(t)

    assert kernel_ns(162) <= 2.0 * kernel_ns(60)
