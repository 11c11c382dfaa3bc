"""Contraction plans with more result blocks than the block pass scans itself when the
host reads the count first (2048): outer products just below and above the 8192 block
pairs from which it does.  The first is scanned by the last workgroup of the block pass in
many chunks, the others by a kernel of its own.  Block list, offsets and tasks must equal
the oracle's exactly (qtensor::operator*, qtensor.cpp:523-734), values agree to 1e-12
relative Frobenius error."""
import numpy as np
import pytest

from test_gpu_contract import check_contract, sec
from ttgpu.flat import INWARD, LINK, OUTWARD, make_index, random_tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nA,nB", [(91, 90), (91, 91), (400, 25)])
def test_outer_product(nA, nB):
    rng = np.random.default_rng(nA)
    idx = [make_index(arrow, name, LINK, 0, sec(range(n), np.ones(n, int)))
           for arrow, name, n in ((INWARD, "a", nA), (OUTWARD, "b", nA), (INWARD, "c", nB), (OUTWARD, "d", nB))]
    oC, _ = check_contract(random_tensor(idx[:2], rng), random_tensor(idx[2:], rng))
    assert oC.nblocks == nA * nB
