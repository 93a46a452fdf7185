"""Key tables of every cell width (2 to 250 log bins a decade range; the coarsest cells that keep the
edges apart are taken) and 1D histograms of 16 and of 32 copies (calls from 1e8 pairs on), against the
oracle and against the binary64 kernel."""
import numpy as np
import pytest

import _oracle
from test_gpu_parity import MAG, TOL, check, field, gpu_hist

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geometry,D", [("flat", 2), ("flat", 3), ("deg", 2)])
@pytest.mark.parametrize("nd", [1, 3, 11, 40, 120, 250])
def test_cell_widths(ctx, geometry, D, nd):
    x, u, _ = field(geometry, D, 1500, nd)
    top = np.pi if geometry == "deg" else np.sqrt(D)
    for edges in (np.geomspace(1e-3, top, nd + 1), np.linspace(0.0, top / 3, nd + 1),
                  np.append(np.geomspace(0.05, 0.06, nd + 1), np.inf)):
        os_, oc, oa, og = _oracle.hist(x, u, edges, op=(0, 2, 0), geometry=geometry, nthreads=4, with_mag=True)
        for prec in ("fp64", "mixed"):
            gs, gc = gpu_hist(ctx, x, u, edges, (0, 2, 0), geometry=geometry, prec=prec)
            check(gs, gc, os_, oc, oa, TOL[prec], f"{geometry} D={D} nd={nd} {prec}", og=og, mag=MAG[prec])


@pytest.mark.parametrize("nd", [1, 20, 33, 100])
def test_copies(ctx, nd):
    x, u, _ = field("flat", 2, 15001, 7)
    edges = np.geomspace(1e-3, np.sqrt(2), nd + 1)
    s64, c64 = gpu_hist(ctx, x, u, edges, (0, 2, 0), prec="fp64")
    sm, cm = gpu_hist(ctx, x, u, edges, (0, 2, 0), prec="mixed")
    ctx.set_tuning(copies=16)
    s16, c16 = gpu_hist(ctx, x, u, edges, (0, 2, 0), prec="mixed")
    ctx.set_tuning()
    assert np.array_equal(c64, cm) and np.array_equal(c64, c16)
    assert np.all(np.abs(sm - s16) <= 1e-12 * np.abs(s16))
    assert np.all(np.abs(sm - s64) <= 1e-6 * np.abs(s64))
