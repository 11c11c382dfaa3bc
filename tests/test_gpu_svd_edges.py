"""Sector SVD (ttg_svd) at the sector sizes where the Jacobi solver changes:
the edges of its 16, 32 and 64 wide forms, one row, and the first sizes of the
block Jacobi, all as sectors of one tensor, against numpy.

The sectors' singular values lie in [1/2, 1], so the Gram matrix loses no more
than a factor of 4, and an eigenpair is off by the rounding of the rotations
that touch it: at most 63 per sweep and 15 sweeps (127 for the block Jacobi's
largest sector here) at 2^-53 each, about 2e-13 if all of them added up.
Bound: 1e-12.  With a cutoff, sectors above 64 rows take their vectors as
R^T W Lambda^(-1/2) of the reduced matrix R R^T, whose iteration stops at
elements of 1e-12 sqrt(g_ii g_jj): there an n-row sector's factors are held to
n times that."""
import ctypes as C

import numpy as np
import pytest

from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, FlatTensor, make_index

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 7, 8, 9, 15, 16, 17, 24, 31, 32, 33, 48, 63, 64, 65, 96, 129]


@pytest.mark.parametrize("direction", [T.MOVE_FROM_LEFT, T.MOVE_FROM_RIGHT])
@pytest.mark.parametrize("cutoff", [0.0, 1e-14])
def test_sector_sizes(direction, cutoff):
    rng = np.random.default_rng(17)
    secs = [((2 * q, 0), n) for q, n in enumerate(SIZES)]
    i = make_index(INWARD, "i", LINK, 0, secs)
    j = make_index(OUTWARD, "j", LINK, 0, secs)
    mats = []
    for n in SIZES:
        u, v = (np.linalg.qr(rng.standard_normal((n, n)))[0] for _ in range(2))
        mats.append((u * np.linspace(1.0, 0.5, n)) @ v)
    bq = np.array([[q, q] for q in range(len(SIZES))], np.int32)
    A = T.DTensor.from_flat(FlatTensor([i, j], bq, np.concatenate([m.reshape(-1, order="F") for m in mats])))
    h = [C.c_void_p() for _ in range(3)]
    tr, kept = C.c_double(0), C.c_int64(0)
    T.check(T.lib().ttg_svd(A.h, 1, direction, cutoff, 0, C.byref(h[0]), C.byref(h[1]), C.byref(h[2]),
                            C.byref(tr), C.byref(kept)))
    U, S, V = (T.DTensor(x, []) for x in h)
    assert kept.value == sum(SIZES)
    u, s, v = U.data(), S.data(), V.data()
    o = k = 0
    for n, m in zip(SIZES, mats):
        un, vn = (a[o:o + n * n].reshape(n, n, order="F") for a in (u, v))
        iso = un if direction == T.MOVE_FROM_LEFT else vn.T
        assert np.max(np.abs(s[k:k + n] - np.linspace(1.0, 0.5, n))) < 1e-12, n
        tol = n * 1e-12 if cutoff > 0 and n > 64 else 1e-12
        assert np.linalg.norm(un @ vn - m, 2) < tol, n
        assert np.linalg.norm(iso.T @ iso - np.eye(n), 2) < tol, n
        o, k = o + n * n, k + n
