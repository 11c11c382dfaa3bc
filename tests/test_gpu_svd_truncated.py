"""Accuracy of the sector SVD (ttg_svd) where singular values fall by many decades, so that
those at the cutoff, or the smallest, are near the rounding of the Gram matrix: factors
and values against numpy's SVD of the sector itself.

Tolerance of the kept part.  The rounding dG of the Gram matrix mixes the kept singular vectors c with the
left-out ones d by K = u_c^T dG u_d / (lambda_c - lambda_d) to first order, which moves the kept
part by sqrt(sum K^2 (sigma_c^2 + sigma_d^2)).  That is computed here from the Gram matrix that
numpy rounds (against 80-bit arithmetic).  The device's is rounded by as much, and an
eigensolver that adds no more than as much again stays within twice that: the bound, for
the geometric mean over the sectors.  (A factorisation that leaves out what is below 1e-15 of
the largest diagonal, and does not correct for it, adds two to three times as much.)"""
import ctypes as C

import numpy as np
import pytest

from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, FlatTensor, make_index

pytestmark = pytest.mark.gpu

SIZES = [(17, 20), (24, 64), (33, 33), (40, 25), (48, 48), (60, 90), (64, 64), (64, 40)]


def kept_part(m, direction):
    """the product of the factors, the isometric one, and the number of kept values"""
    n, c = m.shape
    i = make_index(INWARD, "i", LINK, 0, [((0, 0), n)])
    j = make_index(OUTWARD, "j", LINK, 0, [((0, 0), c)])
    A = T.DTensor.from_flat(FlatTensor([i, j], np.array([[0, 0]], np.int32), m.reshape(-1, order="F")))
    h = [C.c_void_p() for _ in range(3)]
    T.check(T.lib().ttg_svd(A.h, 1, direction, 1e-9, 0, C.byref(h[0]), C.byref(h[1]), C.byref(h[2]),
                            C.byref(C.c_double(0)), C.byref(C.c_int64(0))))
    u, s, v = (T.DTensor(x, []).data() for x in h)
    u, v = u.reshape(n, len(s), order="F"), v.reshape(len(s), c, order="F")
    return u @ v, (u if direction == T.MOVE_FROM_LEFT else v.T), len(s)


def rounding_effect(m, U, S, p):
    """what rounding m m^T to 64 bits moves the part of the first p singular vectors by"""
    x = m.astype(np.longdouble)
    dg = (m @ m.T - x @ x.T).astype(float)
    full = np.linalg.qr(np.hstack([U, np.eye(len(m))]))[0]   # U and the rest of the space
    full[:, :U.shape[1]] = U
    sig = np.concatenate([S, np.zeros(len(m) - len(S))])
    k = full[:, :p].T @ dg @ full[:, p:] / (sig[:p, None] ** 2 - sig[None, p:] ** 2)
    return np.sqrt((k ** 2 * (sig[:p, None] ** 2 + sig[None, p:] ** 2)).sum())


@pytest.mark.parametrize("direction", [T.MOVE_FROM_LEFT, T.MOVE_FROM_RIGHT])
@pytest.mark.parametrize("decades", [9, 13, 20])
def test_kept_part(direction, decades):
    rng = np.random.default_rng(decades)
    ratios = []
    for n, c in SIZES * 3:
        k = min(n, c)
        u, v = (np.linalg.qr(rng.standard_normal((x, k)))[0] for x in (n, c))
        m = (u * np.logspace(0, -decades, k)) @ v.T
        got, iso, p = kept_part(m, direction)
        U, S, V = np.linalg.svd(m, full_matrices=False)
        off = np.linalg.norm(got - (U[:, :p] * S[:p]) @ V[:p])
        if direction == T.MOVE_FROM_LEFT:
            ratios.append(off / rounding_effect(m, U, S, p))
        else:
            ratios.append(off / rounding_effect(m.T, V.T, S, p))
        assert np.linalg.norm(iso.T @ iso - np.eye(p), 2) < 1e-13, (n, c, p)
    assert np.exp(np.mean(np.log(ratios))) < 2.0


@pytest.mark.parametrize("n,c", [(40, 20), (64, 50), (130, 65), (300, 150), (300, 200)])
@pytest.mark.parametrize("decades", [2, 3.5, 3.9])
def test_values_of_sectors_with_a_null_space(n, c, decades):
    """more rows than columns, no cutoff: the singular values down to the smallest, whose
    squares are near 1e-8 of the largest.  The Gram matrix's rounding moves a value by
    u_c^T dG u_c / (2 sigma_c), and an iteration of some eight sweeps that rounds it anew in each
    by eight times that; the largest values by the n roundings of each sweep, halved by the root"""
    for seed in range(3):
        rng = np.random.default_rng(seed)
        u, v = (np.linalg.qr(rng.standard_normal((x, c)))[0] for x in (n, c))
        m = (u * np.logspace(0, -decades, c)) @ v.T
        i = make_index(INWARD, "i", LINK, 0, [((0, 0), n)])
        j = make_index(OUTWARD, "j", LINK, 0, [((0, 0), c)])
        A = T.DTensor.from_flat(FlatTensor([i, j], np.array([[0, 0]], np.int32), m.reshape(-1, order="F")))
        h = [C.c_void_p() for _ in range(3)]
        T.check(T.lib().ttg_svd(A.h, 1, T.MOVE_FROM_LEFT, 0.0, 0, C.byref(h[0]), C.byref(h[1]), C.byref(h[2]),
                                C.byref(C.c_double(0)), C.byref(C.c_int64(0))))
        _, s, _ = (T.DTensor(x, []).data() for x in h)
        U, S, _ = np.linalg.svd(m, full_matrices=False)
        x = m.astype(np.longdouble)
        dg = (m @ m.T - x @ x.T).astype(float)
        moved = np.abs(np.einsum("ic,ij,jc->c", U, dg, U) / (2 * S)).max()
        assert np.abs(s - S).max() < 8 * moved + 8 * n * 2.0 ** -53 / 2, (seed, moved)
