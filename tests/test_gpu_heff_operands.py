"""H_eff products written over one of the operator's own operands (ttg_heff_apply accepts
any y with x's block list): the operand is read to the end before it is written, so the
result is that of a product into a vector of its own, bit for bit."""
import numpy as np
import pytest

from test_gpu_heff import TOL
from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, make_index, random_tensor

pytestmark = pytest.mark.gpu

# matrices of one block list: y = L x W R
PAIRS = [[(1, 0)], [(1, 0)], [(1, 0)]]


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("prec", [T.FP64, T.FP32, T.BF16X3])
def test_product_over_an_operand(prec, which):
    rng = np.random.default_rng(7)
    secs = [((q, 0), d) for q, d in zip(range(-2, 3), [3, 17, 33, 20, 1])]
    i, j = make_index(INWARD, "i", LINK, 0, secs), make_index(OUTWARD, "j", LINK, 0, secs)
    flat = [random_tensor([i, j], rng) for _ in range(4)]
    L, W, R, x = (T.DTensor.from_flat(t) for t in flat)
    h = T.Heff(L, W, R, x, PAIRS, prec)
    y = h.new_output()
    h.apply(x, y)
    want = y.data()
    blocks = [t.to_dense() for t in flat]
    ref = blocks[0] @ blocks[3] @ blocks[1] @ blocks[2]
    assert np.linalg.norm(y.to_flat().to_dense() - ref) <= TOL[prec] * np.linalg.norm(ref)
    out = (L, W, R)[which]
    h.apply(x, out)
    assert np.array_equal(out.data(), want)
