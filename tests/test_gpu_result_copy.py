"""tensor_to_host around the size up to which a kernel writes the result to pinned memory:
single bytes, sizes that are no whole words, data that starts off a word, both sides of the
limit, and results read right after the operator that writes them."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4, 1023, 4096, (256 << 10) - 1, 256 << 10, (256 << 10) + 1])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_result_copy_bytes(hip, n, offset):
    data = np.random.default_rng(n).integers(0, 256, n + offset).astype(np.uint8)
    whole = hip.dev_from(data, O.U8)
    part = hip.lib.tensor_wrap_device(whole.contents.data + offset, (ctypes.c_int * 1)(n), 1, O.U8)
    try:
        assert np.array_equal(hip.dev_read(part, O.U8), data[offset:])
    finally:
        hip.lib.free_tensor(part)
        hip.lib.free_tensor(whole)


def test_result_follows_its_operator(hip):
    """The copy is ordered after the call that writes the tensor, every time."""
    L = hip.lib
    a = hip.dev_from(np.full((4, 1000), 2, np.float32), O.F32)
    y = hip.dev_empty((4, 1000), O.F32)
    L.add_forward(a, a, y)
    for k in range(20):
        L.add_forward(a, y, y)
        assert np.all(hip.dev_read(y, O.F32) == 4 + 2 * (k + 1))
    L.free_tensor(a)
    L.free_tensor(y)
