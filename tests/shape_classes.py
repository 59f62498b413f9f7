"""CPU reference of the level-set derivatives (test infrastructure): the corners of a sphere's box
move by +h and -h in 216 classes 6 apart in every direction, each move a whole oracle geometry
(oscillation fix, fractions, volumes, operator, right-hand side), and a corner's derivative is the sum
of (F_i(+) - F_i(-)) / 2h over the cells c + [-2, 3]^3 with F_i = J_i + lambda_i (b_i - (A p)_i).
Differences of fractions, coefficients and right-hand sides are taken before they meet p and lambda."""
import ctypes as C

import numpy as np

import oracle_py as O

FLUID = 11111111
EQ = 1e-5  # the fix touches corners above it


def corners(w):
    """Coordinates of the upper corners (uniform widths; x stepped from the first box cell)."""
    cell = [float(a[0]) for a in w]
    N, M, K = (len(a) for a in w)
    x0 = (1 + 0.5) * cell[0] + 0.5 * cell[0]
    x = np.concatenate([[0.0], np.add.accumulate(np.r_[x0, np.full(N - 2, cell[0])])])
    return x, (np.arange(M) + 0.5) * cell[1] + 0.5 * cell[1], (np.arange(K) + 0.5) * cell[2] + 0.5 * cell[2]


def raw_sphere(w, center, r):
    """Level set r - |x - c| at the upper corners inside the default box, 0 outside."""
    x, y, z = corners(w)
    N, M, K = (len(a) for a in w)
    qx, qy, qz = (x - center[0])[None, None, :], (y - center[1])[None, :, None], (z - center[2])[:, None, None]
    phi = np.zeros((K, M, N))
    inside = np.s_[:, 1:M - 1, 1:N - 1]
    phi[inside] = (r - np.sqrt(qx * qx + qy * qy + qz * qz))[inside]
    return phi


def moved(phi, cls, step):
    K, M, N = phi.shape
    a, b, c = cls % 6, cls // 6 % 6, cls // 36
    out = phi.copy()
    for y in range(1, M - 1):
        if y % 6 == b:
            for x in range(1, N - 1):
                if x % 6 == a:
                    out[c::6, y, x] += step
    return out


def _shift(a, axis, d):
    """a at the neighbour d = +-1 along an axis (0 past the ends)."""
    b = np.zeros_like(a)
    to, fro = [slice(None)] * 3, [slice(None)] * 3
    to[axis], fro[axis] = (slice(None, -1), slice(1, None)) if d > 0 else (slice(1, None), slice(None, -1))
    b[tuple(to)] = a[tuple(fro)]
    return b


def oscillation_fix(phi):
    """(level set after the fix, passes until one changes nothing): lower neighbours fixed, upper ones not."""
    K, M, N = phi.shape
    box = np.zeros(phi.shape, bool)
    box[:, 1:M - 1, 1:N - 1] = True
    mid = box.copy()
    mid[0] = mid[-1] = False
    cur, passes = phi.copy(), 0
    while True:
        passes += 1
        f = phi.copy()
        for axis, where in ((2, box), (1, box), (0, mid)):
            lo, up = _shift(cur, axis, -1), _shift(phi, axis, 1)
            f = np.where(where & (f > EQ) & (lo < 0) & (up < 0), 0.5 * (lo + up), f)
        if np.array_equal(f, cur, equal_nan=True):
            return cur, passes
        cur = f


def newly_fixed(phi, h):
    """Nodes that some class's move makes the fix touch and that it leaves alone unmoved."""
    base, passes = oscillation_fix(phi)
    count, most = 0, passes
    for cls in range(216):
        for s in (h, -h):
            m = moved(phi, cls, s)
            f, p = oscillation_fix(m)
            count += int(((f != m) & (base == phi)).sum())
            most = max(most, p)
    return passes, most, count


def _geometry(w, phi):
    L = O.lib()
    L.lsxo_geom_build_level_set.argtypes = [C.c_void_p, C.c_void_p] + [C.c_int] * 4
    g = O.Geometry(*w)
    N, M, _ = g.dims
    flat = np.ascontiguousarray(phi, np.float64).ravel()
    if L.lsxo_geom_build_level_set(g.h, flat.ctypes.data, 1, N - 1, 1, M - 1) != 0:
        raise RuntimeError(L.lsxo_last_error().decode())
    return g


def class_gradient(w, phi, p, lam, flow, h):
    """(derivative per corner, bound of its summation's rounding per corner)."""
    K, M, N = phi.shape
    area = (w[1][None, :] * w[2][:, None])[:, :, None]  # dy dz
    P = p.reshape(K, M, N)
    box = np.zeros(phi.shape, bool)
    box[:, 1:M - 1, 1:N - 1] = True
    out, tol = np.zeros(phi.shape), np.zeros(phi.shape)
    for cls in range(216):
        gs = [_geometry(w, moved(phi, cls, s)) for s in (h, -h)]
        f = [g.fields() for g in gs]
        tx = [q["thx"].reshape(K, M, N) for q in f]
        cut = [(q["type"].reshape(K, M, N) > 0) & (q["type"].reshape(K, M, N) != FLUID) & box for q in f]
        west = [np.concatenate([np.zeros((K, M, 1)), t[:, :, :-1]], 2) for t in tx]
        both = ((west[0] - west[1]) - (tx[0] - tx[1])) * area * P
        one = [np.where(c, (a - t) * area * P, 0.0) for c, a, t in zip(cut, west, tx)]
        dJ = np.where(cut[0] & cut[1], both, one[0] - one[1])
        A = gs[0].laplace().to_scipy() - gs[1].laplace().to_scipy()
        b = O.pressure_rhs(gs[0], **flow) - O.pressure_rhs(gs[1], **flow)
        dF = (dJ.ravel() + lam * (b - A @ p)) / (2 * h)
        size = (np.abs(dJ).ravel() + np.abs(lam) * (np.abs(b) + abs(A) @ np.abs(p))) / (2 * h)
        # at most 216 terms a corner, each a sum of at most 9 products: 240 roundings of the size's sum
        for src, dst, scale in ((dF, out, 1.0), (size, tol, 240 * 2.0 ** -53)):
            pad = np.zeros((K + 5, M + 5, N + 5))
            pad[2:2 + K, 2:2 + M, 2:2 + N] = src.reshape(K, M, N)
            acc = np.zeros(phi.shape)
            for k in range(6):
                for j in range(6):
                    for i in range(6):
                        acc += pad[k:k + K, j:j + M, i:i + N]
            z, y, x = np.indices(phi.shape)
            mine = box & (x % 6 + 6 * (y % 6) + 36 * (z % 6) == cls)
            dst[mine] = scale * acc[mine]
    return out, tol
