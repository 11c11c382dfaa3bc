"""Vector operations of the Krylov loop at the edges of their kernels: dot
products around the sizes where the number of workgroups and the unrolled walk
change, the small eigensolver over its whole range of sizes, and an operator
product written over its own input."""
import numpy as np
import pytest

from test_gpu_heff import build_case, run_heff
from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, make_index, random_tensor

pytestmark = pytest.mark.gpu

EPS = 2.3e-16


# 256 elements a workgroup, 512 workgroups, eight strides unrolled
@pytest.mark.parametrize("n", [1, 63, 257, 131071, 131073, 8 * 131072 - 1, 8 * 131072 + 257, 3000001])
def test_dot(n):
    rng = np.random.default_rng(n)
    i = make_index(INWARD, "i", LINK, 0, [((0, 0), n)])
    j = make_index(OUTWARD, "j", LINK, 0, [((0, 0), 1)])
    x, y = random_tensor([i, j], rng), random_tensor([i, j], rng)
    a, b = T.DTensor.from_flat(x), T.DTensor.from_flat(y)
    va, vb = a.data(), b.data()
    assert va.size == n
    want = float(np.sum(va.astype(np.longdouble) * vb))
    # every addition on the longest way to the result rounds once
    tol = (n / 131072 + 32) * EPS * np.abs(va * vb).sum()
    got = [a.dot(b) for _ in range(3)]
    assert abs(got[0] - want) <= tol
    assert got[0] == got[1] == got[2]   # a fixed order of additions
    nrm = float(np.sqrt(np.sum(va.astype(np.longdouble) ** 2)))
    assert abs(a.norm() - nrm) <= (n / 131072 + 32) * EPS * nrm


@pytest.mark.parametrize("n", range(1, 17))
def test_small_eigh(n):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    A = A + A.T
    A[: n // 2, n // 2 :] = A[n // 2 :, : n // 2] = 0   # some pairs need no rotation
    ev, V = T.small_eigh(A)
    # rotations of 6 sweeps of n columns, each to a few units in the last place
    tol = 6 * n * 4 * EPS * np.linalg.norm(A)
    assert np.abs(ev - np.linalg.eigvalsh(A)).max() <= tol
    assert np.abs(A @ V - V * ev).max() <= tol
    assert np.abs(V.T @ V - np.eye(n)).max() <= 6 * n * 4 * EPS


@pytest.mark.parametrize("prec", [T.FP64, T.FP32, T.BF16X3])
def test_product_over_its_input(prec):
    case = build_case("nn_chain", 5, 40, 4, 2.0)
    h, dx, y = run_heff(case, prec)
    if dx.info()[2] != y.info()[2]:
        pytest.skip("the product has more blocks than the vector")
    want = y.data()
    h.apply(dx, dx)
    assert np.array_equal(dx.data(), want)
