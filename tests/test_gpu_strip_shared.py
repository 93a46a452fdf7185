"""B-strips of fields with three components on the sphere: the radial component of every operator that
uses it, where the slices share one position array (column-major positions, which no conversion copies)."""
import numpy as np
import pytest

import sfamd
from test_gpu_strip import check_fields, strips_on  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sf,op", [(sfamd.S2SF, (1, 0, 0)), (sfamd.T2SF, (0, 0, 2)), (sfamd.L2SF, (0, 2, 0))])
def test_radial_component(sf, op):
    rng = np.random.default_rng(16)
    x = np.asfortranarray(np.stack([rng.uniform(-180, 180, 700), np.degrees(np.arcsin(rng.uniform(-1, 1, 700)))]))
    u = rng.normal(size=(3, 700, 3)) * np.array([1.0, 1.0, 5.0])[:, None, None]
    e = np.geomspace(1e-2, 3.1, 14)
    r = sfamd.calculate_structure_function(sf, x, u, e, backend=sfamd.MI355XBackend(precision="mixed"),
                                           count_eltype=np.uint64, distance_metric=sfamd.Haversine(1.0),
                                           output_type=sfamd.StructureFunctionSumsAndCounts)
    check_fields(r, x, u, e, op, "deg", "mixed", f"{op}")
