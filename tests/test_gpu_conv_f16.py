"""float16 Conv2d on the f16 matrix cores against the oracle (tensor_ops.c:1036-1114): every
tile shape and the k split, channel counts around the 8-channel chunks and groups, taps around
the 64-k tiles, odd and even planes (both load widths, every store width), strides, dilations,
asymmetric pads, f16 / f32 outputs and biases.  Products of halves are exact in f32 and the
sums f32, so the tolerance is assert_close's: one unit in the last place of f16, 1e-5 for f32."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_close

pytestmark = pytest.mark.gpu

# name, x shape, M, (KH, KW), pads, strides, dilations, group
CASES = [
    ("c1_group1_m17", (1, 1, 9, 9), 17, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), 1),
    ("c3_stem", (2, 3, 30, 26), 20, (7, 7), (3, 3, 3, 3), (2, 2), (1, 1), 1),
    ("c7", (1, 7, 12, 12), 9, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), 1),
    ("c9_odd_plane", (3, 9, 7, 9), 33, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), 1),
    ("c64_1x1", (2, 64, 16, 16), 65, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1), 1),
    ("c72_split", (1, 72, 14, 14), 70, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), 1),
    ("c512_split_7x7", (1, 512, 7, 7), 40, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), 1),
    ("s2_asym_dil", (2, 20, 21, 23), 24, (3, 2), (2, 0, 1, 3), (2, 3), (2, 1), 1),
    ("group2", (2, 24, 10, 10), 14, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), 2),
    ("group5_c3", (2, 15, 11, 6), 10, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), 5),
    ("tiles_64x128", (8, 16, 56, 56), 72, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), 1),
    ("tiles_128x128", (24, 8, 54, 52), 130, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1), 1),
    ("oh_odd_width2", (2, 16, 10, 5), 8, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), 1),
    # few products per output over many pixels: the general kernel
    ("few_products", (8, 9, 98, 95), 7, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1), 1),
    ("few_products_stride2", (8, 16, 190, 191), 16, (1, 1), (0, 0, 0, 0), (2, 2), (1, 1), 1),
    # many k-tiles through the rings of LDS slots: every remainder of three slots (18, 19 and
    # 20 tiles of 64x128) and of two (2 and 11 tiles of 128x128)
    ("ring_64x128_18", (32, 128, 28, 28), 128, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), 1),
    ("ring_64x128_19", (8, 48, 56, 56), 72, (5, 5), (2, 2, 2, 2), (1, 1), (1, 1), 1),
    ("ring_64x128_20", (8, 136, 56, 56), 72, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), 1),
    ("ring_128x128_2", (24, 120, 54, 52), 130, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1), 1),
    ("ring_128x128_11", (24, 72, 54, 52), 130, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1), 1),
]


@pytest.mark.parametrize("odt,bdt", [(O.F16, O.F32), (O.F16, O.F16), (O.F32, None)], ids=["f16", "f16_bias16", "f32_nobias"])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_conv_f16(hip, oracle_lib, case, odt, bdt):
    name, xs, m, k, pads, strides, dil, group = case
    rng = np.random.default_rng(xs[1] + m)
    x = rng.normal(0, 1, xs).astype(np.float16)
    kg = xs[1] // group * k[0] * k[1]
    w = rng.normal(0, 1 / np.sqrt(kg), (m, xs[1] // group) + k).astype(np.float16)
    b = rng.normal(0, 0.5, (m,)).astype(np.float16 if bdt == O.F16 else np.float32) if bdt is not None else None
    with hip.poisoned():
        y = hip.conv(x, O.F16, w, O.F16, b, bdt or O.F32, odt, list(pads), list(strides), list(dil), group)
    if xs[0] * xs[2] * xs[3] > 5000:          # the last image covers a tile's remainder
        keep = slice(xs[0] - 1, xs[0])
        x, y = x[keep], y[keep]
    ref = oracle_lib.conv(x, O.F16, w, O.F16, b, bdt or O.F32, odt, list(pads), list(strides), list(dil), group)
    assert_close(y, ref, odt, what=name)


def test_conv_f16_nonfinite(hip, oracle_lib):
    """Infinities and NaN in X and W, padding against non-finite weights, f16 overflow."""
    rng = np.random.default_rng(3)
    x = rng.normal(0, 1, (2, 12, 9, 8)).astype(np.float16)
    w = rng.normal(0, 0.2, (10, 12, 3, 3)).astype(np.float16)
    x[0, 3, 4, 4], x[1, 0, 0, 0] = np.inf, np.nan
    w[2, 5, 0, 0], w[7, 1, 2, 2] = np.nan, -np.inf
    w[4] = 6e4
    b = np.zeros(10, np.float32)
    args = ([1, 1, 1, 1], [1, 1], [1, 1], 1)
    y = hip.conv(x, O.F16, w, O.F16, b, O.F32, O.F16, *args)
    ref = oracle_lib.conv(x, O.F16, w, O.F16, b, O.F32, O.F16, *args)
    keep = [m for m in range(10) if m != 4]
    assert_close(y[:, keep], ref[:, keep], O.F16, what="nonfinite")
    # channel 4 sums to beyond f16: the same infinities
    assert np.array_equal(np.isinf(y[:, 4]), np.isinf(ref[:, 4]))


@pytest.mark.parametrize("odt", [O.F16, O.F32], ids=["f16", "f32"])
@pytest.mark.parametrize("sub", ["x", "w", "y"])
def test_conv_f16_subnormals(hip, oracle_lib, sub, odt):
    """Subnormal halves in X or in W count with their value, and subnormal results are rounded
    to the subnormals' spacing."""
    rng = np.random.default_rng(17)
    tiny = lambda shape: (rng.integers(-1023, 1024, shape) * 2.0 ** -24).astype(np.float16)
    xs, ws = (2, 24, 9, 8), (10, 24, 3, 3)
    x = tiny(xs) if sub == "x" else rng.normal(0, 0.02 if sub == "y" else 1, xs).astype(np.float16)
    w = tiny(ws) if sub == "w" else rng.normal(0, 5e-5 if sub == "y" else 1, ws).astype(np.float16)
    args = ([1, 1, 1, 1], [1, 1], [1, 1], 1)
    y = hip.conv(x, O.F16, w, O.F16, None, O.F32, odt, *args)
    ref = oracle_lib.conv(x, O.F16, w, O.F16, None, O.F32, odt, *args)
    assert_close(y, ref, odt, what=sub)
    assert np.count_nonzero(ref) > ref.size // 2


@pytest.mark.parametrize("h,w", [(0, 8), (7, 0)])
@pytest.mark.parametrize("group", [1, 16], ids=["c16", "depthwise"])
def test_conv_f16_of_no_pixels(hip, oracle_lib, h, w, group):
    """No rows or columns, outputs from padding alone: the bias."""
    rng = np.random.default_rng(h)
    x = np.zeros((1, 16, h, w), np.float16)
    wt = rng.normal(0, 1, (16, 16 // group, 3, 3)).astype(np.float16)
    b = rng.normal(0, 1, 16).astype(np.float32)
    with hip.poisoned():
        y = hip.conv(x, O.F16, wt, O.F16, b, O.F32, O.F16, [2, 2, 2, 2], [1, 1], [1, 1], group)
    assert y.size and np.array_equal(y.view(np.float16), np.broadcast_to(b.astype(np.float16)[:, None, None], y.shape))
