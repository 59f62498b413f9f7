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
