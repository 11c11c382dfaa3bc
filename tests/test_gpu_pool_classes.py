"""Device pool: a buffer whose size is a size class (a power of two, or a multiple of an
eighth of the next one) takes that much of the budget and no more, although every buffer is
followed by readable bytes."""
import ctypes as C

import pytest

from ttgpu import lib as T
from ttgpu.flat import INWARD, LINK, OUTWARD, make_index

pytestmark = pytest.mark.gpu


def in_use():
    n = C.c_size_t(0)
    T.check(T.lib().ttg_mem_info(C.byref(n), None, None))
    return n.value


@pytest.mark.parametrize("doubles", [1 << 20, 5 << 18, 1 << 25, 7 << 22])
def test_a_size_class_is_taken_as_it_is(doubles):
    i = make_index(INWARD, "i", LINK, 0, [((0, 0), doubles)])
    j = make_index(OUTWARD, "j", LINK, 0, [((0, 0), 1)])
    T.DTensor.init_blocks([i, j])   # (tables of the first call)
    T.check(T.lib().ttg_finalize())   # no cached buffer of another size to take
    before = in_use()
    x = T.DTensor.init_blocks([i, j])
    assert 8 * doubles <= in_use() - before <= 8 * doubles + 65536   # and the block tables
    del x
