"""Sector SVD (ttg_svd) of graded matrices: columns of a well-conditioned matrix scaled by
factors that fall over many decades, as the tensor of a site has them once it has taken
up its neighbour's singular values (qtt.cpp:821-850).  Without a cutoff every singular
value is kept, and the small ones carry their own relative accuracy.

Tolerance.  With A = B D, D diagonal, the relative error of an eigenvalue of the Gram matrix
D (B^T B) D is at most that of B^T B, componentwise, over its smallest eigenvalue (Demmel and
Veselic, 1992): n roundings (2^-53) in the product and in each of some eight sweeps, times
the squared condition number of B with columns of unit length, halved by the root.  The
reference is a one-sided Jacobi iteration in 80-bit arithmetic."""
import ctypes as C

import numpy as np
import pytest

from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, FlatTensor, make_index

pytestmark = pytest.mark.gpu


def one_sided(A):
    """singular values and right vectors of a column-graded A, descending"""
    n = A.shape[1]
    order = np.argsort(-(A ** 2).sum(0))
    A, V = A[:, order].astype(np.longdouble), np.eye(n, dtype=np.longdouble)[:, order]
    for _ in range(30):
        off = False
        for i in range(n - 1 + n % 2):        # rounds of disjoint pairs
            m1 = n - 1 + n % 2
            pq = [((i, m1) if k == 0 else ((i + k) % m1, (i - k) % m1)) for k in range((m1 + 1) // 2)]
            pq = [(min(p), max(p)) for p in pq if max(p) < n]
            p, q = np.array([x[0] for x in pq]), np.array([x[1] for x in pq])
            a, b, c = (A[:, p] ** 2).sum(0), (A[:, q] ** 2).sum(0), (A[:, p] * A[:, q]).sum(0)
            on = np.abs(c) > 1e-18 * np.sqrt(a * b)
            off |= bool(on.any())
            th = (b - a) / np.where(on, 2 * c, 1)
            t = np.where(on, np.where(th >= 0, 1, -1) / (np.abs(th) + np.sqrt(th * th + 1)), 0)
            cs = 1 / np.sqrt(t * t + 1)
            for M in (A, V):
                x, y = M[:, p].copy(), M[:, q].copy()
                M[:, p], M[:, q] = cs * x - t * cs * y, t * cs * x + cs * y
        if not off:
            break
    s = np.sqrt((A ** 2).sum(0))
    o = np.argsort(-s.astype(float))
    return s[o], V[:, o]


@pytest.mark.parametrize("direction", [T.MOVE_FROM_LEFT, T.MOVE_FROM_RIGHT])
@pytest.mark.parametrize("n,decades", [(12, 10), (12, 20), (16, 14), (24, 14), (32, 10), (40, 6), (40, 10), (40, 14),
                                       (60, 10), (64, 6), (64, 14), (64, 20), (80, 6), (80, 12), (130, 8)])
def test_graded_columns(n, decades, direction):
    rng = np.random.default_rng(n + decades)
    B = rng.standard_normal((3 * n, n))
    B /= np.linalg.norm(B, axis=0)
    m = B * np.logspace(0, -decades, n)
    S, V = one_sided(m)
    # the isometric side is the graded one: V when moving left, U of the transposed when moving right
    a = m if direction == T.MOVE_FROM_RIGHT else np.ascontiguousarray(m.T)
    i = make_index(INWARD, "i", LINK, 0, [((0, 0), a.shape[0])])
    j = make_index(OUTWARD, "j", LINK, 0, [((0, 0), a.shape[1])])
    A = T.DTensor.from_flat(FlatTensor([i, j], np.array([[0, 0]], np.int32), a.reshape(-1, order="F")))
    h = [C.c_void_p() for _ in range(3)]
    T.check(T.lib().ttg_svd(A.h, 1, direction, 0.0, 0, C.byref(h[0]), C.byref(h[1]), C.byref(h[2]),
                            C.byref(C.c_double(0)), C.byref(C.c_int64(0))))
    un, s, vn = (T.DTensor(x, []).data() for x in h)
    assert len(s) == n
    iso = vn.reshape(n, n, order="F").T if direction == T.MOVE_FROM_RIGHT else un.reshape(n, n, order="F")
    tol = 9 * n * 2.0 ** -53 * np.linalg.cond(B) ** 2 / 2
    assert np.abs(s / S - 1).max() < tol
    # vectors: the same over the least relative gap of neighbouring values (2 in the squares)
    gap = float((1 - S[1:] / S[:-1]).min())
    overlap = np.abs((iso * V).sum(0) / np.sqrt((V ** 2).sum(0)) / np.sqrt((iso.astype(np.longdouble) ** 2).sum(0)))
    assert np.sqrt(np.maximum(0, 2 * (1 - overlap))).max() < 4 * n * tol / gap + 1e-9
