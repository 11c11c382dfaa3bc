"""Every work shape of the grouped GEMM gives the oracle's contraction
(qtensor::operator*, qtensor.cpp:523-734) on blocks at the edges of the shapes:
rows, columns and k of 1, one below and above a fragment (16), a 16-byte load's
elements, a tile and a k-tile, with either operand stored either way round; and
the shapes that test_gpu_tiles.py does not list on its contractions.
Tolerances as there: FP64 1e-12, FP32 2e-6, split-BF16 2e-5 relative Frobenius
error."""
import numpy as np
import pytest

from test_gpu_tiles import env_pattern, long_k, mpo_pattern, run, sec
from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, make_index, random_tensor

pytestmark = pytest.mark.gpu

SHAPES = 14   # every work shape; 12 and 13 came after test_gpu_tiles.py's list


def edges(rng):
    """A(i, k) * B(k, j) with every pairing of row, column and k counts"""
    ds = [1, 15, 16, 17, 31, 33, 47, 49, 63, 65]
    i = make_index(INWARD, "i", LINK, 0, sec(range(0, 20, 2), ds))
    k = make_index(OUTWARD, "k", LINK, 0, sec(range(0, 20, 2), ds[::-1]))
    j = make_index(OUTWARD, "j", LINK, 0, sec(range(0, 20, 2), ds[3:] + ds[:3]))
    return random_tensor([i, k], rng), random_tensor([k.dag(), j], rng)


def edges_nk(rng):
    """the same with both operands stored the other way round: B(j, k) and A(k, i)"""
    ds = [1, 15, 16, 17, 31, 33, 47, 49, 63, 65]
    i = make_index(INWARD, "i", LINK, 0, sec(range(0, 20, 2), ds))
    k = make_index(OUTWARD, "k", LINK, 0, sec(range(0, 20, 2), ds[::-1]))
    j = make_index(OUTWARD, "j", LINK, 0, sec(range(0, 20, 2), ds[3:] + ds[:3]))
    return random_tensor([k, i], rng), random_tensor([j, k.dag()], rng)


@pytest.mark.parametrize("cfg", range(SHAPES))
@pytest.mark.parametrize("prec", [T.FP64, T.FP32, T.BF16X3])
@pytest.mark.parametrize("make", [edges, edges_nk])
def test_edges(make, prec, cfg, monkeypatch):
    A, B = make(np.random.default_rng(11))
    run(A, B, prec, cfg, monkeypatch)


@pytest.mark.parametrize("cfg", [12, 13])
@pytest.mark.parametrize("prec", [T.FP64, T.FP32, T.BF16X3])
@pytest.mark.parametrize("make", [env_pattern, mpo_pattern, long_k])
def test_more_shapes(make, prec, cfg, monkeypatch):
    A, B = make(np.random.default_rng(11))
    run(A, B, prec, cfg, monkeypatch)


def test_rows_of_a_large_operand():
    """The vector kernel's items of an operand above 256 MB stand by rows, not by result
    block: every result block against a sum over its tasks."""
    rng = np.random.default_rng(2)
    i = make_index(INWARD, "i", LINK, 0, sec([0, 2], [4000, 3700]))
    j = make_index(INWARD, "j", LINK, 0, sec([0, 2], [1511, 1489]))
    k = make_index(OUTWARD, "k", LINK, 0, sec([0, 2, 4], [2, 1, 2]))
    s = make_index(INWARD, "s", LINK, 0, sec([0, 2], [1, 2]))
    n = make_index(OUTWARD, "n", LINK, 0, sec([0, 2, 4, 6], [2, 3, 1, 2]))
    A, B = random_tensor([i, j, k], rng), random_tensor([k.dag(), s, n], rng)
    assert A.data.nbytes > 256 << 20
    dA, dB = T.DTensor.from_flat(A), T.DTensor.from_flat(B)
    plan = T.Plan(dA, dB, [(2, 0)])
    C = plan.new_output()
    plan.execute(dA, dB, C)
    got, (_, co) = C.data(), C.meta()
    ao, bo = A.block_offsets(), B.block_offsets()
    tasks = plan.tasks()
    assert len({t[0] for t in tasks}) == len(co) - 1
    for c in range(len(co) - 1):
        want = 0.0
        for _, a, b, M, N, K in tasks[tasks[:, 0] == c]:
            want = want + A.data[ao[a]:ao[a + 1]].reshape(M, K, order="F") @ \
                B.data[bo[b]:bo[b + 1]].reshape(K, N, order="F")
        # two products of five terms' sizes at most
        assert np.abs(got[co[c]:co[c + 1]].reshape(want.shape, order="F") - want).max() < 1e-13
