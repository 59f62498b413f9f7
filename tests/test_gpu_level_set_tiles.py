"""The Bezier level set on grids that no tile of 8 x 8 x 4 nodes fills, from boxes inside the grid: equal to
the oracle's bit for bit."""
import numpy as np
import pytest

import oracle_py as O
from test_gpu_geometry import axes_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(33, 31, 30), (39, 26, 29), (17, 24, 13)])
def test_bezier_level_set_of_any_grid(lsx, dims):
    center, axes = (0.45, 0.5, 0.55), (0.25, 0.2, 0.15)
    ctrl = lsx.bezier_perturb(lsx.bezier_ellipsoid(center, axes), 0.01, seed=2)
    w = axes_for(lsx, dims, 1.02)
    ref = O.Geometry(*w).build_bezier(ctrl, center, axes)
    got = lsx.Geometry(*w).build("bezier", center, axes, ctrl=ctrl).fields()
    assert np.array_equal(got["phi"], ref.level_set()["phi"])
    assert np.array_equal(got["type"], ref.fields()["type"])
