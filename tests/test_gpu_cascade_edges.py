"""The cascade's stencil and line passes at the edges of their tiles (16 lines x 64 cells per
wavefront, rows of 64 cells and more by 64 x 4 tiles, lines whose forward result does not fit LDS),
through one application of the one-level preconditioner against the oracle.  The passes run the
reference's operations in the reference's order, so the results are equal bit for bit."""
import numpy as np
import pytest

import oracle_py as O
import problems as P

pytestmark = pytest.mark.gpu

DIMS = [(3, 4, 5), (15, 17, 16), (16, 16, 16), (63, 5, 4), (64, 4, 5), (65, 6, 3), (5, 64, 3), (4, 65, 7), (3, 5, 63),
        (7, 3, 66), (129, 3, 4), (4, 130, 3), (314, 3, 4), (316, 4, 3), (3, 320, 4), (4, 3, 385)]


@pytest.mark.parametrize("dims", DIMS, ids=["x".join(map(str, d)) for d in DIMS])
def test_one_level_application_is_the_oracles(lsx, dims):
    g, A = P.synthetic_cut(*dims, seed=sum(dims))
    S = lsx.MGFGMRES(levels=1)
    S.set(A, np.zeros(A.n), np.zeros(A.n), lsx.Task(eps=1.0))
    v = np.random.default_rng(3).standard_normal(A.n)
    z = S.precondition(v)
    assert np.abs(z).max() > 0
    assert np.array_equal(z, O.Solver(A, eps=1.0, precond="mg1").mg_apply(v))


# 7-point levels of up to 4096 cells and 27-point levels of up to 1024 run in one workgroup, with
# their restrictions, the coarsest LU and the prolongations: whole grids, from level 1, from level 2
SMALL = [(4, 4, 4), (8, 4, 6), (3, 3, 3), (5, 5, 3), (12, 12, 12), (20, 12, 12), (16, 16, 16), (17, 17, 9), (17, 17, 17),
         (9, 5, 33), (20, 20, 20), (24, 24, 24), (40, 24, 24), (33, 33, 33)]


@pytest.mark.parametrize("dims", SMALL, ids=["x".join(map(str, d)) for d in SMALL])
@pytest.mark.parametrize("fix", [False, True])
def test_cascade_application_is_the_oracles(lsx, dims, fix):
    g, A = P.synthetic_cut(*dims, seed=sum(dims))
    S = lsx.MGFGMRES(z_head_fix=fix)
    S.set(A, np.zeros(A.n), np.zeros(A.n), lsx.Task(eps=1.0))
    v = np.random.default_rng(3).standard_normal(A.n)
    z = S.precondition(v)
    S.kernel_timing(True)  # per-level launches
    assert np.array_equal(z, S.precondition(v))
    if not fix:
        assert np.array_equal(z, O.Solver(A, eps=1.0).mg_apply(v))
