"""Device copies of a tensor's data around the size from which the runtime makes them
(64 MiB) and at odd lengths below it: the same bytes, and independent of the source."""
import numpy as np
import pytest

from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, make_index

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 100001, (1 << 23) - 1, 1 << 23, (1 << 23) + 1])
def test_copy(n):
    i = make_index(INWARD, "i", LINK, 0, [((0, 0), n)])
    j = make_index(OUTWARD, "j", LINK, 0, [((0, 0), 1)])
    a = T.DTensor.init_blocks([i, j])
    x = np.random.default_rng(n).standard_normal(n)
    a.upload(x)
    b = a.copy()
    a.fill(0.0)
    assert np.array_equal(b.data(), x)
