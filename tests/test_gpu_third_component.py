"""A third velocity component that is not finite: every operator of the reference takes it (times zero
where the value does not depend on it), so a bin's sum is NaN or infinite where one of its pairs has such a
point.  Against the oracle's pairs."""
import numpy as np
import pytest

import _oracle
from test_gpu_parity import field, gpu_hist

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geometry", ["flat", "deg"])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -1e308])
@pytest.mark.parametrize("op", [(0, 1, 0), (0, 2, 0), (0, 3, 0), (0, 0, 1), (0, 0, 2), (0, 0, 3), (0, 1, 1), (1, 0, 0),
                                (2, 0, 0)])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_third_component(ctx, geometry, bad, op, prec):
    x, u, edges = field(geometry, 3, 90, 31)
    n = 90
    u[2, 17] = bad
    u[2, 60] = -bad
    if np.isfinite(bad):  # one pair, whose difference overflows (sums of more would by their order)
        n, x, u = 2, x[:, [17, 60]], u[:, [17, 60]]
    want = np.zeros(len(edges) - 1)
    cnt = np.zeros(len(edges) - 1, dtype=np.uint64)
    with np.errstate(invalid="ignore", over="ignore"):
        for i in range(n):
            for j in range(i + 1, n):
                ok, _, v, db, _ = _oracle.pair(x, u, edges, i, j, op=op, geometry=geometry)
                if ok and 1 <= db < len(edges):
                    want[db - 1] += v
                    cnt[db - 1] += 1
    gs, gc = gpu_hist(ctx, x, u, edges, op, geometry=geometry, prec=prec)
    gs, gc = gs.reshape(-1), gc.reshape(-1)
    assert np.array_equal(gc, cnt)
    assert np.array_equal(np.isnan(gs), np.isnan(want)) and np.array_equal(np.isinf(gs), np.isinf(want))
