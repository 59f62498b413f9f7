"""The V-cycle's fused launches against the launches one by one, bit for bit: red-black levels with
all sweeps of a side in one launch of 16^3 regions (levels of up to 64^3 cells), and the small levels
in one workgroup, forward and transposed.  Sizes: one cell past a tile of 8 or 12, exact tiles, odd
axes, the largest level taken, an x axis of three cells, a coarsest level with its dense inverse; one and
two sweeps a side, a_p from the faces or read, operators with and without a diagonal of their own."""
import numpy as np
import pytest

import problems as P

pytestmark = pytest.mark.gpu

DIMS = [(33, 17, 25), (40, 24, 16), (37, 50, 21), (64, 64, 64), (3, 48, 26), (40, 3, 24), (24, 37, 12)]


@pytest.mark.parametrize("precision", ["mixed", "mixed16", "fp64-vcycle"])
@pytest.mark.parametrize("dims", DIMS)
def test_fused_levels_are_bitwise(lsx, dims, precision):
    g, A = P.body_free(*dims) if min(dims) < 8 else P.synthetic_cut(*dims, seed=11)
    v = P.random_rhs(g, seed=12, A=A)
    w = np.random.default_rng(4).standard_normal(A.n) * (A.to_scipy().diagonal() < 0)
    for n_pre, n_post in ((2, 2), (1, 2), (2, 1)):
        for diag in (True, False):
            z = []
            for fuse in (True, False):
                S = lsx.solver("fgmres", precision, fused_sweep=int(fuse), coarse_fuse=fuse, diag_faces=diag)
                S.set(A, np.zeros(A.n), np.zeros(A.n), lsx.mixed_task(1.0, n_pre=n_pre, n_post=n_post))
                z.append((S.precondition(v), S.precondition_transpose(w), S.precondition(w)))
            for a, c in zip(*z):
                assert np.linalg.norm(a) > 0 and np.array_equal(a, c), (n_pre, n_post, diag, np.abs(a - c).max())
    print(f"dims={dims} precision={precision} levels={S.num_levels()}", flush=True)
