"""The level-set derivative of bodies of a few cells, where the oscillation fix moves nodes: phi =
r - |x - c| has dphi/dr = 1 at every corner, so the corners' derivatives add up to that of the
Lagrangian F = J + lambda . (b - A p) with the radius, here by central differences of whole
geometries (p and lambda fixed, differences of b, A p and J before they meet lambda).  The radius
step is 1e-6 of a cell: F is smooth while no type changes, so the difference's own error is of the
order of its square, and 1e-5, the bound of the other shape tests, is kept."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [0.95, 1.1, 1.6, 2.3, 4.2])
@pytest.mark.parametrize("dims", [(18, 16, 17), (12, 20, 13)], ids=["18x16x17", "12x20x13"])
def test_radius_derivative_of_small_spheres(lsx, dims, cells):
    w = [np.full(n, 1.0 / n) for n in dims]
    cell = 1.0 / min(dims)
    center, r = (0.53, 0.46, 0.51), cells * cell
    rng = np.random.default_rng(int(10 * cells))
    sizes = lsx.face_sizes(*dims)
    p, lam = rng.standard_normal(sizes[3]), rng.standard_normal(sizes[3])
    flow = dict(u=1.0 + rng.uniform(-0.05, 0.05, sizes[0]), v=rng.uniform(-0.05, 0.05, sizes[1]),
                w=rng.uniform(-0.05, 0.05, sizes[2]))

    def parts(radius):
        g = lsx.Geometry(*w).build("sphere", center, (radius,))
        S = lsx.MGFGMRES(levels=1)
        S.set_geometry(g, None, None, lsx.Task(eps=1.0))
        return g, g.fields()["type"], g.drag(p)[0], g.pressure_rhs(**flow) - S.apply_operator(p)

    g, t0, _, _ = parts(r)
    gphi, _ = g.shape_gradient(p, lam, lsx.OBJ_DRAG_X, flow=flow, ctrl=False)
    h = 1e-6 * cell
    _, tp, Jp, rp = parts(r + h)
    _, tm, Jm, rm = parts(r - h)
    assert np.array_equal(tp, tm)
    if not np.any((t0 > 0) & (t0 != 11111111)):  # the sphere lies between the corners
        assert not gphi.any()
        return
    ref = ((Jp - Jm) + lam @ (rp - rm)) / (2 * h)
    scale = np.abs(gphi).sum()
    print(f"dims={dims} cells={cells} sum={gphi.sum():.6e} ref={ref:.6e} scale={scale:.3e}", flush=True)
    assert scale > 0
    assert abs(gphi.sum() - ref) <= 1e-5 * scale
