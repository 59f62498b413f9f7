"""Shape gradient of a body whose level set is NaN at some corners (one control point so large that the
closest-point search overflows) while the oscillation fix chains at others: the call returns, and its
derivatives are those of whole geometries, NaN where theirs are."""
import numpy as np
import pytest

import oracle_py as O
import shape_classes as SC

DIMS = (12, 12, 12)
# centre, semi-axis, patch, value of its control point (1, 2): NaN at corners whose direction is that of
# a patch's edge, where the search starts on the edge
BODIES = [((0.5, 0.5, 0.5416666666666666), 0.22421074673411492, 0, -1.7e308),
          ((0.4166666666666667, 0.4583333333333333, 0.4166666666666667), 0.18411070721906256, 1, 1.7e308),
          ((0.5833333333333334, 0.4583333333333333, 0.5), 0.12345596070793989, 1, 1.7e308)]


def overflowing(center, axis, patch, value):
    ctrl = O.bezier_ellipsoid(center, (axis,) * 3)
    ctrl[patch, 1, 2, :] = value
    w = [np.full(n, 1.0 / n) for n in DIMS]
    x, y, z = SC.corners(w)
    pts = np.stack(np.meshgrid(z, y, x, indexing="ij")[::-1], -1).reshape(-1, 3)
    N, M, K = DIMS
    phi = np.zeros((K, M, N))
    inside = np.s_[:, 1:M - 1, 1:N - 1]
    phi[inside] = O.bezier_phi(ctrl, center, (axis,) * 3, pts).reshape(K, M, N)[inside]
    return w, ctrl, phi


@pytest.mark.parametrize("center,axis,patch,value", BODIES)
def test_bodies_have_nan_and_a_chain(center, axis, patch, value):
    _, _, phi = overflowing(center, axis, patch, value)
    _, passes = SC.oscillation_fix(phi)
    assert passes > 2 and np.isnan(phi).any() and (phi > 0).any()


@pytest.mark.gpu
@pytest.mark.parametrize("center,axis,patch,value", BODIES)
def test_gradient_returns(lsx, center, axis, patch, value):
    w, ctrl, phi = overflowing(center, axis, patch, value)
    rng = np.random.default_rng(7)
    sizes = lsx.face_sizes(*DIMS)
    p, lam = rng.standard_normal(sizes[3]), rng.standard_normal(sizes[3])
    flow = dict(u=1.0 + rng.uniform(-0.05, 0.05, sizes[0]), v=rng.uniform(-0.05, 0.05, sizes[1]),
                w=rng.uniform(-0.05, 0.05, sizes[2]))
    g = lsx.Geometry(*w).build("bezier", center, (axis,) * 3, ctrl=ctrl)
    assert np.array_equal(g.fields()["phi"], SC.oscillation_fix(phi)[0].ravel(), equal_nan=True)
    gphi, _ = g.shape_gradient(p, lam, lsx.OBJ_DRAG_X, flow=flow, ctrl=False)
    ref, tol = SC.class_gradient(w, phi, p, lam, flow, 1e-7 * min(float(a[0]) for a in w))
    ref, tol = ref.ravel(), tol.ravel()
    fin = np.isfinite(ref)
    print(f"NaN nodes {int(np.isnan(phi).sum())} derivatives: NaN {int(np.isnan(ref).sum())} finite != 0 "
          f"{int((ref[fin] != 0).sum())}", flush=True)
    assert np.array_equal(np.isnan(gphi), np.isnan(ref))
    assert np.all(np.abs(gphi[fin] - ref[fin]) <= tol[fin])
