"""f32 convolutions of a few images (64x64 tiles, with and without slices of k) against the
oracle (tensor_ops.c:1036-1114), plain and with the fused epilogue, whose bits are the
separate calls'; tolerance assert_close's 1e-5 for f32 sums."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_bitexact, assert_close

pytestmark = pytest.mark.gpu

# x shape, M, stride, group
CASES = [((1, 64, 56, 56), 128, 2, 1), ((1, 256, 14, 14), 160, 2, 1), ((2, 512, 7, 7), 130, 1, 1), ((1, 16, 9, 9), 20, 1, 1),
         ((1, 64, 20, 20), 300, 1, 2), ((3, 48, 17, 13), 129, 1, 1)]


@pytest.mark.parametrize("xs,m,stride,group", CASES, ids=["x".join(map(str, c[0])) + f"-{c[1]}" for c in CASES])
def test_conv_small_grid(hip, oracle_lib, xs, m, stride, group):
    rng = np.random.default_rng(m)
    x = rng.normal(0, 1, xs).astype(np.float32)
    kg = xs[1] // group * 9
    w = rng.normal(0, 1 / np.sqrt(kg), (m, xs[1] // group, 3, 3)).astype(np.float32)
    b = rng.normal(0, 0.5, (m,)).astype(np.float32)
    args = ([1, 1, 1, 1], [stride, stride], [1, 1], group)
    with hip.poisoned():
        y = hip.conv(x, O.F32, w, O.F32, b, O.F32, O.F32, *args)
    assert_close(y, oracle_lib.conv(x, O.F32, w, O.F32, b, O.F32, O.F32, *args), O.F32, what="conv")
    skip = rng.normal(0, 1, y.shape).astype(np.float32)
    seq = hip.binary("add", hip.unary("relu", y, O.F32, O.F32), O.F32, skip, O.F32, O.F32)
    assert_bitexact(hip.conv_fused(x, w, b, skip, 1, O.F32, *args), seq, O.F32, what="epilogue")
