"""Sector SVD (ttg_svd) without a cutoff when device allocations are refused: large
sectors then go the way that needs less memory, and the call either succeeds, with the
right factors and no error left behind, or reports the refusal."""
import ctypes as C

import numpy as np
import pytest

from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, FlatTensor, make_index

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cutoff", [0.0, 1e-9])
def test_refused_allocations(cutoff):
    n = 130
    rng = np.random.default_rng(3)
    u, v = (np.linalg.qr(rng.standard_normal((n, n)))[0] for _ in range(2))
    m = (u * np.linspace(1.0, 0.5, n)) @ v
    i = make_index(INWARD, "i", LINK, 0, [((0, 0), n)])
    j = make_index(OUTWARD, "j", LINK, 0, [((0, 0), n)])
    A = T.DTensor.from_flat(FlatTensor([i, j], np.array([[0, 0]], np.int32), m.reshape(-1, order="F")))
    lib = T.lib()
    assert lib.ttg_svd(None, 1, 0, 0.0, 0, None, None, None, None, None) != 0   # leaves its own message
    before = lib.ttg_last_error()
    outcome = []
    for k in range(1, 61):   # more than the call makes
        h = [C.c_void_p() for _ in range(3)]
        T.check(lib.ttg_pool_fail_after(k))
        rc = lib.ttg_svd(A.h, 1, T.MOVE_FROM_LEFT, cutoff, 0, C.byref(h[0]), C.byref(h[1]), C.byref(h[2]),
                         C.byref(C.c_double(0)), C.byref(C.c_int64(0)))
        message = lib.ttg_last_error()
        T.check(lib.ttg_pool_fail_after(0))
        outcome.append(rc)
        if rc:
            assert b"refused" in message or b"allocation failed" in message, k
            assert lib.ttg_svd(None, 1, 0, 0.0, 0, None, None, None, None, None) != 0
            continue
        assert message == before, k
        un, s, vn = (T.DTensor(x, []).data() for x in h)
        un, vn = un.reshape(n, n, order="F"), vn.reshape(n, n, order="F")
        # the singular values lie in [1/2, 1]: the bound of the sector sizes' test
        assert np.abs(s - np.linspace(1.0, 0.5, n)).max() < 1e-12, k
        assert np.linalg.norm(un @ vn - m, 2) < 1e-12, k
        assert np.linalg.norm(un.T @ un - np.eye(n), 2) < 1e-12, k
    assert outcome[0] and not outcome[-1]
    last = max(k for k, rc in enumerate(outcome) if rc)
    # without a cutoff some refusals are answered with the other solver; with one, none
    assert (0 in outcome[:last]) == (cutoff == 0.0)
