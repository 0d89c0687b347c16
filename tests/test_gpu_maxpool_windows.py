"""f32 MaxPool windows on LDS row tiles and the direct 2x2 kernel against the oracle
(tensor_ops.c:1116-1165), bit for bit: every window and stride, planes of less than one strip,
several planes per block, several row tiles per plane, outputs that reach past the input, with
NaN, +-0, -inf and windows wholly in the padding."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_bitexact

pytestmark = pytest.mark.gpu

# x shape, window, stride, pads
CASES = [((1, 1, 1, 1), 3, 1, (1, 1, 1, 1)), ((3, 70, 7, 7), 3, 1, (1, 1, 1, 1)), ((2, 900, 5, 6), 3, 2, (1, 1, 1, 1)),
         ((2, 3, 150, 131), 3, 1, (1, 1, 1, 1)), ((2, 5, 57, 55), 3, 2, (1, 1, 1, 1)), ((2, 5, 58, 56), 3, 2, (0, 0, 0, 0)),
         ((2, 3, 21, 21), 5, 1, (2, 2, 2, 2)), ((1, 4, 100, 64), 5, 2, (2, 2, 2, 2)), ((2, 3, 17, 18), 2, 1, (0, 0, 1, 1)),
         ((2, 3, 17, 18), 2, 2, (1, 1, 1, 1)), ((2, 3, 18, 18), 2, 2, (0, 0, 0, 0)), ((2, 7, 19, 17), 2, 2, (0, 0, 0, 0)),
         ((1, 5, 33, 1026), 2, 2, (0, 0, 0, 0)), ((1, 2, 9, 1000), 3, 1, (1, 1, 1, 1)), ((1, 3, 6, 6), 3, 2, (4, 4, 4, 4)),
         ((2, 3, 18, 19), 2, 2, (0, 0, 1, 1))]
# wide planes, enough of them for the row tiles: several tiles per plane and chunks per row
TILES = [((8, 20, 150, 131), 3, 1, (1, 1, 1, 1)), ((2, 65, 57, 55), 3, 2, (1, 1, 1, 1)), ((2, 65, 58, 56), 3, 2, (0, 0, 0, 0)),
         ((1, 66, 100, 64), 5, 2, (2, 2, 2, 2)), ((1, 260, 9, 1000), 3, 1, (1, 1, 1, 1)), ((4, 600, 20, 130), 2, 2, (1, 1, 1, 1)),
         ((3, 100, 70, 75), 2, 1, (0, 0, 0, 0))]
CASES += TILES


@pytest.mark.parametrize("shape,k,s,pads", CASES, ids=["x".join(map(str, c[0])) + f"_k{c[1]}s{c[2]}p{c[3][0]}{c[3][2]}" for c in CASES])
def test_maxpool_windows(hip, oracle_lib, shape, k, s, pads):
    rng = np.random.default_rng(sum(shape))
    x = rng.normal(0, 1, shape).astype(np.float32)
    flat = x.reshape(-1)
    for value in (np.nan, -0.0, 0.0, -np.inf, np.inf):
        flat[rng.choice(flat.size, max(1, flat.size // 40), replace=False)] = value
    x[..., : shape[2] // 2, : shape[3] // 2] = np.where(x[..., : shape[2] // 2, : shape[3] // 2] > 0, 0.0, -0.0)
    with hip.poisoned():
        y = hip.maxpool(x, O.F32, O.F32, [k, k], list(pads), [s, s])
    assert_bitexact(y, oracle_lib.maxpool(x, O.F32, O.F32, [k, k], list(pads), [s, s]), O.F32, what=f"maxpool {shape}")
