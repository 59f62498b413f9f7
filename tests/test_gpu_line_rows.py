"""Line relaxation on rows that no multiple of four or eight cells fill, and y and z lines of full and
partial segments of eight cells: one sweep on the finest level against the exact line solves on the
oracle's CSR operator, and the cycle against its transpose.  Tolerances: the line systems of cubic
cells are diagonally dominant (two of six couplings on the line), so a solve carries a few dozen
roundings, 2^-53 and 2^-24 each: 1e-12 and 2e-5 leave a factor of ten."""
import numpy as np
import pytest

import problems as P
from test_gpu_smoothers import ref_line_sweep

pytestmark = pytest.mark.gpu

# N: CPL 4 and two lines a wavefront (65..128), CPL 4 (129..256), CPL 8 (257..512), remainders 1, 2, 3, 5;
# M, K: 1 to 14 segments, full and partial
DIMS = [(65, 9, 12), (66, 16, 5), (127, 8, 17), (128, 7, 9), (129, 24, 6), (191, 5, 33), (261, 6, 16), (260, 9, 8),
        (33, 111, 7), (20, 23, 64)]


@pytest.mark.parametrize("precision,tol", [("fp64-vcycle", 1e-12), ("mixed", 2e-5)])
@pytest.mark.parametrize("dims", DIMS)
def test_line_sweep_of_any_row(lsx, dims, precision, tol):
    g, A = P.body_free(*dims, L=tuple(n / 32.0 for n in dims))
    S = lsx.solver("fgmres", precision, smoother="line")
    S.set(A, np.zeros(A.n), np.zeros(A.n), lsx.mixed_task(1.0))
    act = A.to_scipy().diagonal() < 0
    rng = np.random.default_rng(3)
    b, x0, y = (rng.standard_normal(A.n) * act for _ in range(3))
    e = []
    for zero in (False, True):
        x = S.smooth(b, x0, sweeps=1, zero_guess=zero)
        ref = ref_line_sweep(A, dims, b, np.zeros(A.n) if zero else x0)
        e.append(np.linalg.norm(x - ref) / np.linalg.norm(ref))
    Bx, BTy = S.precondition(b), S.precondition_transpose(y)
    t = abs(Bx @ y - b @ BTy) / (np.linalg.norm(Bx) * np.linalg.norm(y))
    print(f"dims={dims} precision={precision} rel err {e[0]:.3e} from zero {e[1]:.3e} transpose {t:.3e}", flush=True)
    assert max(e) <= tol and t <= tol


@pytest.mark.parametrize("precision", ["fp64-vcycle", "mixed"])
@pytest.mark.parametrize("dims", [(33, 28, 24), (32, 32, 32), (18, 13, 11), (100, 30, 10), (17, 5, 32), (40, 24, 33)])
def test_small_line_levels_in_one_launch_are_bitwise(lsx, dims, precision):
    """The one-workgroup cycle over small line-relaxed levels gives the bits of the launches one by
    one, forward and transposed: y and z lines of one and two segments, x lines of up to 50 cells."""
    g, A = P.synthetic_cut(*dims, seed=11)
    act = A.to_scipy().diagonal() < 0
    rng = np.random.default_rng(3)
    v, w = (rng.standard_normal(A.n) * act for _ in range(2))
    for n_pre, n_post in ((2, 2), (1, 2), (2, 1), (3, 1)):
        z = []
        for fuse in (True, False):
            S = lsx.solver("fgmres", precision, smoother="line", coarse_fuse=fuse)
            S.set(A, np.zeros(A.n), np.zeros(A.n), lsx.mixed_task(1.0, n_pre=n_pre, n_post=n_post))
            z.append((S.precondition(v), S.precondition_transpose(w), S.precondition(w)))
        for a, c in zip(*z):
            assert np.linalg.norm(a) > 0 and np.array_equal(a, c), (n_pre, n_post, np.abs(a - c).max())
    print(f"dims={dims} precision={precision} levels={S.num_levels()}", flush=True)
