"""Sector SVD (ttg_svd) of sectors whose rank is below their size, with and
without a cutoff: the pivoted Cholesky factorisation ahead of the Jacobi
iteration ends at the rank, on the edges of the solver's widths, and without a
cutoff a sector that needs more vectors than its rank goes the plain way.

The nonzero singular values lie in [1/2, 1].  The factorisation leaves a remainder of
n roundings (2^-53) of the largest diagonal, and an eigenpair is off by that over
the smallest nonzero eigenvalue, 1/4: 300 x 4 x 1.1e-16 = 1.3e-13 at the largest
sector here.  Bound: 1e-12; orthonormality, which the last step restores to n
roundings, 1e-13 with a cutoff and 1e-12 (the rotations' own) without."""
import ctypes as C

import numpy as np
import pytest

from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, FlatTensor, make_index

pytestmark = pytest.mark.gpu

# (rows, columns, rank)
SMALL = [(16, 16, 5), (17, 17, 1), (17, 30, 16), (33, 20, 17), (48, 64, 32), (64, 64, 33), (64, 10, 10), (64, 64, 64),
         (63, 63, 15), (20, 20, 0)]


def svd(secs, direction, cutoff, K=0):
    rng = np.random.default_rng(5)
    i = make_index(INWARD, "i", LINK, 0, [((2 * q, 0), n) for q, (n, _, _) in enumerate(secs)])
    j = make_index(OUTWARD, "j", LINK, 0, [((2 * q, 0), c) for q, (_, c, _) in enumerate(secs)])
    mats = []
    for n, c, r in secs:
        u, v = np.linalg.qr(rng.standard_normal((n, n)))[0], np.linalg.qr(rng.standard_normal((c, c)))[0]
        mats.append((u[:, :r] * np.linspace(1.0, 0.5, r)) @ v[:r])
    bq = np.array([[q, q] for q in range(len(secs))], np.int32)
    A = T.DTensor.from_flat(FlatTensor([i, j], bq, np.concatenate([m.reshape(-1, order="F") for m in mats])))
    h = [C.c_void_p() for _ in range(3)]
    tr, kept = C.c_double(0), C.c_int64(0)
    T.check(T.lib().ttg_svd(A.h, 1, direction, cutoff, K, C.byref(h[0]), C.byref(h[1]), C.byref(h[2]),
                            C.byref(tr), C.byref(kept)))
    U, S, V = (T.DTensor(x, []) for x in h)
    qu, ou = U.meta()
    _, ov = V.meta()
    out, s, k0 = {}, S.data(), 0
    u, v = U.data(), V.data()
    for b, (q, _) in enumerate(qu):
        n, c, _ = secs[q]
        k = int(ou[b + 1] - ou[b]) // n
        out[int(q)] = (u[ou[b]:ou[b + 1]].reshape(n, k, order="F"), s[k0:k0 + k],
                       v[ov[b]:ov[b + 1]].reshape(k, c, order="F"))
        k0 += k
    return mats, out, kept.value


def check(secs, direction, cutoff):
    mats, out, kept = svd(secs, direction, cutoff)
    assert kept == sum(r if cutoff else min(n, c) for n, c, r in secs)
    for q, ((n, c, r), m) in enumerate(zip(secs, mats)):
        if cutoff and r == 0:
            assert q not in out
            continue
        u, s, v = out[q]
        iso = u if direction == T.MOVE_FROM_LEFT else v.T
        k = r if cutoff else min(n, c)
        assert len(s) == k
        assert np.abs(s[:r] - np.linspace(1.0, 0.5, r)).max(initial=0) < 1e-12, (n, c, r)
        # a zero singular value is the root of a rounding of the Gram matrix
        assert np.all(s[r:] < np.sqrt(300 * 2.3e-16)), (n, c, r)
        assert np.linalg.norm(u @ v - m, 2) < 1e-12, (n, c, r)
        tol = 1e-13 if cutoff else 1e-12
        assert np.linalg.norm(iso.T @ iso - np.eye(k), 2) < tol, (n, c, r)


@pytest.mark.parametrize("direction", [T.MOVE_FROM_LEFT, T.MOVE_FROM_RIGHT])
@pytest.mark.parametrize("cutoff", [0.0, 1e-10])
def test_small_sectors(direction, cutoff):
    check(SMALL, direction, cutoff)


def test_kept_values_within_the_rank():
    """without a cutoff but with a limit on the values, a sector of lower rank than size
    can serve every value asked for"""
    mats, out, kept = svd([(60, 60, 30), (64, 64, 40)], T.MOVE_FROM_LEFT, 0.0, K=20)
    assert kept == 20
    s = np.sort(np.concatenate([x[1] for x in out.values()]))[::-1]
    want = np.sort(np.concatenate([np.linspace(1, 0.5, 30), np.linspace(1, 0.5, 40)]))[::-1][:20]
    assert np.abs(s - want).max() < 1e-12
    for u, _, _ in out.values():
        assert np.linalg.norm(u.T @ u - np.eye(u.shape[1]), 2) < 1e-13


LARGE = [(65, 65, 30), (65, 65, 65), (100, 40, 40), (128, 128, 64), (130, 200, 127), (200, 300, 200), (300, 300, 150),
         (300, 150, 90), (70, 70, 1), (80, 80, 0)]


@pytest.mark.parametrize("direction", [T.MOVE_FROM_LEFT, T.MOVE_FROM_RIGHT])
@pytest.mark.parametrize("cutoff", [0.0, 1e-10])
def test_large_sectors(direction, cutoff):
    check(LARGE, direction, cutoff)


@pytest.mark.parametrize("cutoff", [0.0, 1e-10])
def test_equal_diagonals(cutoff):
    """more equal remaining diagonals than a panel has candidates"""
    n = 150
    i = make_index(INWARD, "i", LINK, 0, [((0, 0), n)])
    j = make_index(OUTWARD, "j", LINK, 0, [((0, 0), n)])
    A = T.DTensor.from_flat(FlatTensor([i, j], np.array([[0, 0]], np.int32), 3.0 * np.eye(n).reshape(-1)))
    h = [C.c_void_p() for _ in range(3)]
    T.check(T.lib().ttg_svd(A.h, 1, T.MOVE_FROM_LEFT, cutoff, 0, C.byref(h[0]), C.byref(h[1]), C.byref(h[2]),
                            C.byref(C.c_double(0)), C.byref(C.c_int64(0))))
    u, s, v = (T.DTensor(x, []).data() for x in h)
    u, v = u.reshape(n, n, order="F"), v.reshape(n, n, order="F")
    assert np.abs(s - 3.0).max() < 1e-12
    assert np.abs(u @ v - 3.0 * np.eye(n)).max() < 1e-12
