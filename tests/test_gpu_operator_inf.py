"""Operator products of a vector with an infinite value at cells of the grid's border: a row takes the
neighbours that are there and nothing in place of the others, so that it is infinite, not NaN, where its
terms are.  Seven-point rows of a symmetric and of an unsymmetric matrix, 27-point rows of the levels
below; the terms of a row in ascending column order, bit for bit."""
import numpy as np
import pytest

import oracle_py as O
import problems as P

pytestmark = pytest.mark.gpu

OFFS = [(i % 3 - 1, i // 3 % 3 - 1, i // 9 - 1) for i in range(27)]
SEVEN = [OFFS[q] for q in (4, 10, 12, 13, 14, 16, 22)]


def product(planes, dims, x):
    N, M, K = dims
    x = x.reshape(K, M, N)
    y = np.zeros((K, M, N))
    for a, (i, j, k) in zip(planes, SEVEN if len(planes) == 7 else OFFS):
        to = tuple(slice(max(0, -o), n - max(0, o)) for o, n in ((k, K), (j, M), (i, N)))
        fro = tuple(slice(max(0, o), n - max(0, -o)) for o, n in ((k, K), (j, M), (i, N)))
        y[to] = y[to] + a.reshape(K, M, N)[to] * x[fro]
    return y.ravel()


def vector(dims, where):
    N, M, K = dims
    x = np.random.default_rng(5).standard_normal(N * M * K)
    cell = {"corner": (0, 0, 0), "far-corner": (N - 1, M - 1, K - 1), "edge": (0, M // 2, K - 1),
            "face": (N // 2, M - 1, K // 2), "west": (0, M // 2, K // 2)}[where]
    x[cell[0] + N * (cell[1] + M * cell[2])] = np.inf
    return x


@pytest.mark.parametrize("where", ["corner", "far-corner", "edge", "face", "west"])
@pytest.mark.parametrize("dims", [(16, 16, 16), (64, 16, 16), (17, 9, 17)], ids=["16", "64x16x16", "17x9x17"])
@pytest.mark.parametrize("symmetric", [True, False])
def test_rows_next_to_the_border(lsx, dims, where, symmetric):
    g, A = P.synthetic_cut(*dims, seed=sum(dims))
    if not symmetric:
        val = A.val * np.random.default_rng(2).uniform(0.9, 1.1, A.val.size)
        A = O.Csr(A.dims, A.rowptr, A.col, val)
    S = lsx.MGFGMRES()
    S.set(A, np.zeros(A.n), np.zeros(A.n), lsx.Task(eps=1.0))
    for level in (0, 1):
        d = S.level_dims(level)
        planes = S.level_stencil(level)
        x = vector(d, where)
        y, ref = S.apply_operator(x, level), product(planes, d, x)
        print(f"{dims} {where} level {level}: inf {int(np.isinf(ref).sum())} NaN {int(np.isnan(ref).sum())} here NaN "
              f"{int(np.isnan(y).sum())}", flush=True)
        assert np.isinf(ref).any()
        assert np.array_equal(y, ref, equal_nan=True)
