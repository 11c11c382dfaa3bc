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


# list lengths at the ends of 16-byte elements, and above the size that one
# copy launch takes (256 KiB)
@pytest.mark.parametrize("nb", [1, 2, 3, 5, 7, 1023, 1025, 32768, 40001])
def test_block_lists(nb):
    n = max(2, int(np.ceil(np.sqrt(nb))))
    i = make_index(INWARD, "i", LINK, 0, [((q, 0), 1) for q in range(n)])
    j = make_index(OUTWARD, "j", LINK, 0, [((q, 0), 1 + q % 3) for q in range(n)])
    qi = np.array([(b // n, b % n) for b in range(nb)], dtype=np.int32)
    x = random_tensor([i, j], np.random.default_rng(nb), block_qi=qi)
    a, b = T.DTensor.from_flat(x), T.DTensor.from_flat(x)
    assert np.array_equal(np.asarray(a.meta()[0]).reshape(-1, 2), qi)
    assert a.dot(b) == b.dot(a)          # compares the lists
    c = a.copy()
    T.check(T.lib().ttg_tensor_dag(a.h))
    T.check(T.lib().ttg_tensor_dag(a.h))
    assert a.dot(c) == c.dot(c)          # the same structure again
    assert np.array_equal(c.data(), x.data)
    other = qi.copy()
    if nb > 1 and nb < n * n:            # as many blocks, one at another place
        other[-1] = (n - 1, n - 1)
        if tuple(other[-1]) != tuple(qi[-1]) and (n - 1) % 3 == qi[-1][1] % 3:
            d = T.DTensor.from_flat(random_tensor([i, j], np.random.default_rng(1), block_qi=other))
            with pytest.raises(RuntimeError):
                a.dot(d)
    del b, c


def test_dag_outlives_its_source():
    """a flipped structure shares the tables of the one it came from"""
    rng = np.random.default_rng(0)
    i = make_index(INWARD, "i", LINK, 0, [((q, 0), 3) for q in range(40)])
    j = make_index(OUTWARD, "j", LINK, 0, [((q, 0), 2) for q in range(40)])
    x = random_tensor([i, j], rng)
    a = T.DTensor.from_flat(x)
    T.check(T.lib().ttg_tensor_dag(a.h))   # the only holder of the first structure is now the second
    others = [T.DTensor.from_flat(random_tensor([i, j], rng)) for _ in range(50)]
    assert np.array_equal(np.asarray(a.meta()[0]).reshape(-1, 2), x.block_qi)
    del others
