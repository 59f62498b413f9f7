"""Many set-ups on one handle: their device blocks are kept from one to the next, and cycles are captured at
a (input, output) pair's first or second use, as the set-up before used its pairs.  Two operators of
different sizes in turn, one solve each (no pair comes twice: later set-ups run a pair's first cycle
eagerly), then several solves on one set-up (eager, captured, replayed), then a set-up again, all
against handles that set up once and run eagerly, bit for bit."""
import ctypes as C

import numpy as np
import pytest

import problems as P

pytestmark = pytest.mark.gpu


class Handle:
    """One C handle with the options of a solver object, set up any number of times."""

    def __init__(self, lsx, kind, precision, A, **options):
        self.lsx = lsx
        self.S = lsx.solver(kind, precision, **options)
        self.S.set(A, np.zeros(A.n), np.zeros(A.n), lsx.mixed_task(1.0, restart=30, max_it=500))

    def set(self, A):
        N, M, K = A.dims
        L = self.lsx.lib()
        assert L.lsx_set_csr(self.S.h, N, M, K, A.rowptr.ctypes.data, A.col.ctypes.data, A.val.ctypes.data, len(A.val),
                             self.lsx.MEM_HOST) == 0

    def solve(self, b, eps=1e-8):
        L = self.lsx.lib()
        x, it, nr = np.zeros(b.size), C.c_int(), C.c_double()
        assert L.lsx_set_eps(self.S.h, eps * np.linalg.norm(b)) == 0
        assert L.lsx_solve(self.S.h, b.ctypes.data, x.ctypes.data, self.lsx.MEM_HOST, C.byref(it), C.byref(nr)) == 0
        return x, it.value


@pytest.mark.parametrize("kind,precision,options", [("fgmres", "mixed", {}), ("fgmres", "fp64-vcycle", {}),
                                                    ("bicgstab", "mixed", {}), ("fgmres", "mixed", {"smoother": "line"}),
                                                    ("fgmres", "fp64", {})],
                         ids=["fgmres-mixed", "fgmres-fp64", "bicgstab-mixed", "fgmres-line", "cascade"])
def test_set_ups_in_turn(lsx, kind, precision, options):
    problems = [P.synthetic_cut(24, 16, 16, seed=3), P.synthetic_cut(32, 32, 16, seed=4)]
    rhs = [[P.random_rhs(g, seed=s, A=A) for s in (1, 2, 3)] for g, A in problems]
    ref = []
    for (g, A), bs in zip(problems, rhs):
        E = Handle(lsx, kind, precision, A, **options)
        ref.append([E.solve(b) for b in bs])
    graphs = {} if precision == "fp64" else {"graphs": True}
    H = Handle(lsx, kind, precision, problems[0][1], **graphs, **options)
    order = [(0, 1), (1, 1), (0, 1), (1, 1), (0, 1), (1, 3), (0, 1), (0, 1), (1, 1), (0, 3)]
    order += [(k % 2, 1) for k in range(18)]
    for step, (which, solves) in enumerate(order):
        if step:
            H.set(problems[which][1])
        for k in range(solves):
            x, it = H.solve(rhs[which][k])
            xr, itr = ref[which][k]
            assert it == itr and np.array_equal(x, xr), (step, which, k, it, itr, np.abs(x - xr).max())
