"""Contraction planning at the sizes where its kernels change: runs of 64 sorted
keys and their merge, more blocks than one workgroup plans (1024), one and two
host waits, more result blocks than the block pass scans itself (2048) - with block
lists in any order, repeated left and right tuples, and up to five contracted
indices.  Block list, offsets and tasks must equal the oracle's exactly
(qtensor::operator*, qtensor.cpp:523-734), values agree to 1e-12 relative Frobenius
error."""
import numpy as np
import pytest

import oracle as O
from test_gpu_contract import check_contract, sec
from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, SITE, legal_blocks, make_index, random_tensor

pytestmark = pytest.mark.gpu


def some(idx, n, rng):
    """a tensor of n legal blocks of idx, in random order"""
    bq = legal_blocks(idx)
    assert len(bq) >= n, len(bq)
    return random_tensor(idx, rng, block_qi=bq[rng.permutation(len(bq))[:n]])


@pytest.mark.parametrize("nA,nB", [(1, 1), (2, 63), (63, 64), (64, 65), (65, 128), (129, 63), (250, 33), (257, 300),
                                   (512, 513), (1023, 9), (1024, 40), (1025, 9), (9, 1025), (1500, 1300)])
def test_blocks(nA, nB):
    rng = np.random.default_rng(nA + nB)
    i = make_index(INWARD, "i", LINK, 0, sec(range(-40, 41), rng.integers(1, 3, 81)))
    k = make_index(OUTWARD, "k", LINK, 0, sec(range(-30, 31), rng.integers(1, 3, 61)))
    s = make_index(INWARD, "s", SITE, 0, sec(range(-12, 13), np.ones(25, int)))
    j = make_index(OUTWARD, "j", LINK, 0, sec(range(-40, 41), rng.integers(1, 3, 81)))
    t = make_index(INWARD, "t", SITE, 0, sec(range(-12, 13), np.ones(25, int)))
    check_contract(some([i, s, k], nA, rng), some([k.dag(), t, j], nB, rng))


@pytest.mark.parametrize("np_", [1, 2, 3, 4, 5])
def test_pairs(np_):
    """np_ contracted indices in two runs, in B in another order than in A, among free
    ones (a layout of more than two strides per dimension is refused)"""
    rng = np.random.default_rng(np_)
    ks = [make_index((INWARD, OUTWARD)[p % 2], "k%d" % p, LINK, 0, sec([-1, 0, 1], rng.integers(1, 4, 3)))
          for p in range(np_)]
    a = make_index(INWARD, "a", LINK, 0, sec(range(-3, 4), rng.integers(1, 4, 7)))
    b = make_index(OUTWARD, "b", LINK, 0, sec(range(-3, 4), rng.integers(1, 4, 7)))
    c = make_index(OUTWARD, "c", SITE, 0, sec([-1, 1], [1, 2]))
    A = random_tensor([ks[0], a] + ks[1:] + [c], rng, keep=0.6)
    B = random_tensor([k.dag() for k in ks[1:]] + [b, ks[0].dag()], rng, keep=0.6)
    check_contract(A, B)
    check_contract(B, A)


def test_many_result_blocks():
    """an outer product: every pair of blocks with the charge zero is a result block"""
    rng = np.random.default_rng(8)
    a = make_index(INWARD, "a", LINK, 0, sec(range(60), np.ones(60, int)))
    b = make_index(OUTWARD, "b", LINK, 0, sec(range(60), np.ones(60, int)))
    c = make_index(INWARD, "c", LINK, 0, sec(range(45), np.ones(45, int)))
    d = make_index(OUTWARD, "d", LINK, 0, sec(range(45), np.ones(45, int)))
    oC, _ = check_contract(random_tensor([a, b], rng), random_tensor([c, d], rng))
    assert oC.nblocks == 60 * 45
