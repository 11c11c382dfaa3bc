"""Sector SVD (ttg_svd) of tensors of very small and very large entries: the Gram
matrices of these are as far as 1e-280 and 1e280, where the squares of their
elements leave the range of a double.  One sector of every solver (up to 16, 32 and
64 rows, block Jacobi), against numpy on the tensor of unit scale.

The singular values lie in [1/2, 1] of the scale; the bound is the one of the sector
sizes' test, 1e-12: a change of scale by a power of two changes no rounding."""
import ctypes as C

import numpy as np
import pytest

from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, FlatTensor, make_index

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cutoff", [0.0, 1e-9])
@pytest.mark.parametrize("exponent", [-465, -332, -266, -232, 0, 232, 266, 332, 465])
@pytest.mark.parametrize("n", [9, 30, 60, 100])
def test_scaled_tensor(n, exponent, cutoff):
    rng = np.random.default_rng(n)
    u, v = (np.linalg.qr(rng.standard_normal((n, n)))[0] for _ in range(2))
    w = np.linspace(1.0, 0.5, n)
    m = (u * w) @ v
    scale = 2.0 ** exponent
    i = make_index(INWARD, "i", LINK, 0, [((0, 0), n)])
    j = make_index(OUTWARD, "j", LINK, 0, [((0, 0), n)])
    A = T.DTensor.from_flat(FlatTensor([i, j], np.array([[0, 0]], np.int32), (m * scale).reshape(-1, order="F")))
    h = [C.c_void_p() for _ in range(3)]
    T.check(T.lib().ttg_svd(A.h, 1, T.MOVE_FROM_LEFT, cutoff, 0, C.byref(h[0]), C.byref(h[1]), C.byref(h[2]),
                            C.byref(C.c_double(0)), C.byref(C.c_int64(0))))
    un, s, vn = (T.DTensor(x, []).data() for x in h)
    un, vn = un.reshape(n, n, order="F"), vn.reshape(n, n, order="F") / scale
    assert np.abs(s / scale - w).max() < 1e-12
    assert np.linalg.norm(un @ vn - m, 2) < 1e-12
    assert np.linalg.norm(un.T @ un - np.eye(n), 2) < 1e-12
