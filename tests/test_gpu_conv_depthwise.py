"""Depthwise Conv2d (one input channel per group) against the oracle (tensor_ops.c:1036-1114):
windows with strips (3x3, 5x5 at stride 1 and 2) and any other, planes of less than one
strip, several planes per block, several row tiles per plane, rows wider than a wave, channel
multipliers, f16 storage; the fused epilogue and the quantized input bit for bit with the
calls they replace.  The tolerance is the convolution's (assert_close: 1e-5 for f32 sums of
at most 49 terms, one unit in the last place for f16)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_bitexact, assert_close

pytestmark = pytest.mark.gpu

# x shape, channel multiplier, (KH, KW), pads, strides, dilations
CASES = [
    ("one_pixel", (1, 3, 1, 1), 1, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),
    ("7x7_planes", (5, 97, 7, 7), 1, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),
    ("many_small", (40, 64, 6, 5), 1, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),
    ("56", (2, 5, 56, 56), 1, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),
    ("s2_odd", (2, 9, 57, 55), 1, (3, 3), (1, 1, 1, 1), (2, 2), (1, 1)),
    ("tiles_wide", (1, 3, 150, 131), 1, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),
    ("very_wide", (1, 2, 9, 900), 1, (3, 3), (0, 0, 0, 0), (1, 1), (1, 1)),
    ("5x5", (2, 6, 33, 29), 1, (5, 5), (2, 2, 2, 2), (1, 1), (1, 1)),
    ("5x5_s2", (2, 6, 100, 40), 1, (5, 5), (2, 2, 2, 2), (2, 2), (1, 1)),
    ("7x7_window", (1, 4, 20, 22), 1, (7, 7), (3, 3, 3, 3), (1, 1), (1, 1)),
    ("1x1", (2, 8, 9, 9), 1, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1)),
    ("s3_dil2_asym", (2, 4, 31, 27), 1, (3, 2), (2, 0, 1, 3), (3, 2), (2, 3)),
    ("multiplier", (3, 8, 12, 13), 3, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),
    ("one_channel_in", (4, 1, 28, 28), 16, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),
    ("no_pad_edge", (1, 2, 8, 8), 1, (3, 3), (0, 0, 0, 0), (1, 1), (1, 1)),
]


def _data(case, npdt="float32"):
    _, xs, mult, k, pads, strides, dil = case
    rng = np.random.default_rng(sum(xs) + mult)
    x = rng.normal(0, 1, xs).astype(npdt)
    w = rng.normal(0, 1 / np.sqrt(k[0] * k[1]), (xs[1] * mult, 1) + k).astype(npdt)
    b = rng.normal(0, 0.5, (xs[1] * mult,)).astype(np.float32)
    return x, w, b, list(pads), list(strides), list(dil), xs[1]


@pytest.mark.parametrize("dt,odt", [(O.F32, O.F32), (O.F16, O.F16), (O.F16, O.F32)], ids=["f32", "f16", "f16_to_f32"])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_depthwise(hip, oracle_lib, case, dt, odt):
    x, w, b, pads, strides, dil, group = _data(case, "float32" if dt == O.F32 else "float16")
    bias = b if case[0] != "56" else None
    with hip.poisoned():
        y = hip.conv(x, dt, w, dt, bias, O.F32, odt, pads, strides, dil, group)
    assert_close(y, oracle_lib.conv(x, dt, w, dt, bias, O.F32, odt, pads, strides, dil, group), odt, what=case[0])


@pytest.mark.parametrize("case", [CASES[i] for i in (1, 4, 5, 9, 12)], ids=lambda c: c[0])
def test_depthwise_fused(hip, case):
    """Relu and the skip add, fake quantization, and a quantized input: the calls' bits."""
    x, w, b, pads, strides, dil, group = _data(case)
    y = hip.conv(x, O.F32, w, O.F32, b, O.F32, O.F32, pads, strides, dil, group)
    skip = np.random.default_rng(5).normal(0, 1, y.shape).astype(np.float32)
    seq = hip.binary("add", hip.unary("relu", y, O.F32, O.F32), O.F32, skip, O.F32, O.F32)
    assert_bitexact(hip.conv_fused(x, w, b, skip, 1, O.F32, pads, strides, dil, group), seq, O.F32, what="epilogue")
    s, z = np.float32(0.03), np.uint8(120)
    fq = hip.qdq_fused(seq, s, z, s, z, "uint8")
    assert_bitexact(hip.conv_fused_qdq(x, w, b, skip, 1, s, z, s, z, "uint8", pads, strides, dil, group), fq, O.F32,
                    what="fake quantization")
    for dt in (O.U8, O.I8):
        q = np.clip(np.rint(x / 0.02), -128, 127).astype(np.int8)
        q = q if dt == O.I8 else (q.astype(np.int16) + 128).astype(np.uint8)
        zx = np.array([3], q.dtype)
        xd = hip.qdq1("dequantize", q, dt, np.float32(0.02), zx, dt, O.F32)
        want = hip.conv_fused(xd, w, b, skip, 1, O.F32, pads, strides, dil, group)
        got = hip.dq_conv_fused(q, dt, np.float32(0.02), zx, w, b, skip, 1, pads, strides, dil, group)
        assert_bitexact(got, want, O.F32, what="codes")


@pytest.mark.parametrize("value", [np.nan, np.inf], ids=["nan", "inf"])
def test_depthwise_padding_meets_weights(hip, oracle_lib, value):
    """A padded tap is 0 * w: a non-finite weight shows in the border outputs only."""
    x, w, b, pads, strides, dil, group = _data(CASES[3])
    w[1, 0, 0, 0] = value
    y = hip.conv(x, O.F32, w, O.F32, b, O.F32, O.F32, pads, strides, dil, group)
    assert_close(y, oracle_lib.conv(x, O.F32, w, O.F32, b, O.F32, O.F32, pads, strides, dil, group), O.F32, what="w")
