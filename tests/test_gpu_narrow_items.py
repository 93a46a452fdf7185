"""Work items narrower than a row tile (calls too small to fill the device with whole tiles) against
the oracle: sizes at the edges of a 16-column item, of a wave and of a row tile, every kind of
histogram and kernel.  Counts are bit-identical; sums within the bounds of the parity tests, which
hold for any split of the pairs."""
import numpy as np
import pytest

import _oracle
from test_gpu_parity import MAG, TOL, check, field, gpu_hist
from test_gpu_single_pass import check_sp, gpu_sp, row_scales

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geometry,D", [("flat", 2), ("flat", 3), ("deg", 2)])
@pytest.mark.parametrize("n", [2, 17, 65, 257, 1025])
def test_narrow_items(ctx, geometry, D, n):
    x, u, edges = field(geometry, D, max(n, 8), 900 + n)
    x, u = np.ascontiguousarray(x[:, :n]), np.ascontiguousarray(u[:, :n])
    ve = np.linspace(-3, 3, 20)
    for op, v in [((0, 2, 0), None), ((0, 0, 3), None), ((0, 1, 0), ve)]:
        os_, oc, oa, og = _oracle.hist(x, u, edges, op=op, geometry=geometry, vedges=v, nthreads=2, with_mag=True)
        for prec in ("fp64", "mixed", "fixed"):
            if prec == "fixed" and v is None:
                continue
            gs, gc = gpu_hist(ctx, x, u, edges, op, geometry=geometry, vedges=v, prec=prec)
            label = f"{geometry} D={D} n={n} op={op} {prec}"
            if prec == "fixed":  # 2^-23 value-bin widths a pair on top (factor 1.5 spare)
                assert np.array_equal(gc, oc), label
                bound = TOL["mixed"] * oa + MAG["mixed"] * og + 1.5 * 2.0 ** -23 * (ve[1] - ve[0]) * oc.astype(float)
                assert np.all(np.abs(gs - os_) <= bound + 1e-300), label
            else:
                check(gs, gc, os_, oc, oa, TOL[prec], label, og=og, mag=MAG[prec])


@pytest.mark.parametrize("n", [257, 1025])
def test_narrow_items_single_pass(ctx, n):
    x, u, edges = field("flat", 2, n, 950 + n)
    ss, sc = _oracle.single_pass(x, u, edges, nthreads=2)
    oa, og = row_scales(x, u, edges, "flat")
    for prec in ("fp64", "mixed"):
        gs, gc = gpu_sp(ctx, x, u, edges, "flat", prec)
        check_sp(gs, gc, ss, sc, oa, og, prec, f"single pass n={n} {prec}")
