"""The level-set derivative corner by corner, where the oscillation fix is at work: small spheres whose
fix chains (a fixed node reads a fixed node) in the unmoved geometry, only once a corner has moved, or not
at all, and whose moves bring the fix to nodes that it leaves alone unmoved (values within the step
of 0 or of the fix's threshold: bodies aligned with the grid, or a large step).  Against the oracle's
whole geometries; the differences that enter are equal bit for bit, so the bound is the rounding of their
sums."""
import numpy as np
import pytest

import shape_classes as SC

# dims, centre, radius, h_rel; fix passes unmoved > 2, at most moved > 2, nodes fixed only when moved
ALIGNED = (12, 11, 13)
BODIES = {
    "chain": (ALIGNED, (0.5783422140890314, 0.5170325879781816, 0.4942619330363663), 0.21599155144732243, 1e-7,
              True, True, False),
    "chain-and-new": (ALIGNED, (0.48130206734962533, 0.5819917923324593, 0.40861337771364087), 0.2388802898528322, 8e-3,
                      True, True, True),
    "long-chain-and-new": (ALIGNED, (0.5011945268130367, 0.5631020813318023, 0.44341343621442525),
                           0.09616169629389505, 8e-3, True, True, True),
    "chain-and-new-2": (ALIGNED, (0.5368753316141885, 0.5181429463809739, 0.5324255179916482), 0.16860452499390585, 2e-3,
                        True, True, True),
    "aligned": (ALIGNED, (0.333333333333, 0.454545454545, 0.692307692308), 1 / 11, 1e-7, False, True, True),
    "aligned-large-step": (ALIGNED, (0.333333333333, 0.636363636364, 0.230769230769), 1 / 11, 2e-3, False, True, True),
    "new-alone": (ALIGNED, (0.41321649934481497, 0.5682634559224766, 0.4133380017534203), 0.14755008686260573, 8e-3,
                  False, False, True),
    "plain": (ALIGNED, (0.596167057765246, 0.537108396896139, 0.5300918552535633), 0.21324892129081582, 1e-7,
              False, False, False),
}


def body(name):
    dims, center, r, h_rel = BODIES[name][:4]
    w = [np.full(n, 1.0 / n) for n in dims]
    return dims, w, center, r, h_rel, h_rel * min(float(a[0]) for a in w)


@pytest.mark.parametrize("name", list(BODIES))
def test_bodies_are_what_they_stand_for(name):
    _, w, center, r, _, h = body(name)
    passes, most, new = SC.newly_fixed(SC.raw_sphere(w, center, r), h)
    assert (passes > 2, most > 2, new > 0) == BODIES[name][4:], (passes, most, new)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(BODIES))
def test_corner_derivatives_of_moved_geometries(lsx, name):
    dims, w, center, r, h_rel, h = body(name)
    rng = np.random.default_rng(7)
    sizes = lsx.face_sizes(*dims)
    p, lam = rng.standard_normal(sizes[3]), rng.standard_normal(sizes[3])
    flow = dict(u=1.0 + rng.uniform(-0.05, 0.05, sizes[0]), v=rng.uniform(-0.05, 0.05, sizes[1]),
                w=rng.uniform(-0.05, 0.05, sizes[2]))
    g = lsx.Geometry(*w).build("sphere", center, (r,))
    phi = SC.raw_sphere(w, center, r)
    assert np.array_equal(g.fields()["phi"], SC.oscillation_fix(phi)[0].ravel())
    gphi, _ = g.shape_gradient(p, lam, lsx.OBJ_DRAG_X, flow=flow, h_rel=h_rel, ctrl=False)
    ref, tol = SC.class_gradient(w, phi, p, lam, flow, h)
    diff = np.abs(gphi - ref.ravel())
    print(f"{name}: corners {int((ref != 0).sum())} max|ref|={np.abs(ref).max():.3e} max diff={diff.max():.3e} "
          f"over bound {int((diff > tol.ravel()).sum())}", flush=True)
    assert (ref != 0).any()
    assert np.all(diff <= tol.ravel())
