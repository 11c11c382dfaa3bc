"""Sector SVD (ttg_svd) of the widest sectors it accepts (8192 rows), with and without a
cutoff, and one row more, which it refuses.  The singular values lie in [1/2, 1]; the
bound is the one of the sectors of lower rank than size: n roundings (2^-53) of the
largest diagonal over the smallest eigenvalue, 1/4: 8192 x 4 x 1.1e-16 = 3.6e-12."""
import ctypes as C

import numpy as np
import pytest

from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, FlatTensor, make_index

pytestmark = pytest.mark.gpu


def svd(n, c, cutoff):
    rng = np.random.default_rng(1)
    u, v = np.linalg.qr(rng.standard_normal((n, c)))[0], np.linalg.qr(rng.standard_normal((c, c)))[0]
    w = np.linspace(1.0, 0.5, c)
    m = (u * w) @ v
    i = make_index(INWARD, "i", LINK, 0, [((0, 0), n)])
    j = make_index(OUTWARD, "j", LINK, 0, [((0, 0), c)])
    A = T.DTensor.from_flat(FlatTensor([i, j], np.array([[0, 0]], np.int32), m.reshape(-1, order="F")))
    h = [C.c_void_p() for _ in range(3)]
    T.check(T.lib().ttg_svd(A.h, 1, T.MOVE_FROM_LEFT, cutoff, 0, C.byref(h[0]), C.byref(h[1]), C.byref(h[2]),
                            C.byref(C.c_double(0)), C.byref(C.c_int64(0))))
    un, s, vn = (T.DTensor(x, []).data() for x in h)
    return m, w, un.reshape(n, c, order="F"), s, vn.reshape(c, c, order="F")


@pytest.mark.parametrize("cutoff", [0.0, 1e-9])
@pytest.mark.parametrize("n", [8181, 8182, 8192])
def test_widest_sectors(n, cutoff):
    m, w, u, s, v = svd(n, 40, cutoff)
    assert np.abs(s - w).max() < 3.6e-12
    assert np.linalg.norm(u @ v - m) < 40 * 3.6e-12
    assert np.linalg.norm(u.T @ u - np.eye(40), 2) < 3.6e-12


def test_one_row_more():
    with pytest.raises(RuntimeError, match="larger than 8192"):
        svd(8193, 40, 1e-9)
