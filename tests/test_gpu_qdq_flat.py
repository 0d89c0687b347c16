"""QuantizeLinear / DequantizeLinear of lengths and channel runs that are no multiple of four
elements, bit for bit with the oracle (tensor_ops.c:999-1034): one scale, scales along the
first, a middle and the last axis with runs of 1 to 50 elements, lengths of 1 to 3 past a group
of four, zero points of the code type and float32, ties, infinities, NaN, a zero scale."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_bitexact

pytestmark = pytest.mark.gpu

# shape, axis (None: one scale)
CASES = [((1,), None), ((7,), None), ((1026,), None), ((5, 7, 9), 0), ((5, 7, 9), 1), ((5, 7, 9), 2), ((3, 5, 49), 1),
         ((64, 3, 7, 7), 0), ((2, 1, 3), 2), ((1, 9, 1), 1), ((130, 21), 1), ((4, 6, 2), 1), ((33, 50), 0), ((3, 1000), 1)]


@pytest.mark.parametrize("code", [O.U8, O.I8, O.E4M3, O.E5M2], ids=["u8", "i8", "e4m3", "e5m2"])
@pytest.mark.parametrize("zf32", [False, True], ids=["code_zp", "f32_zp"])
@pytest.mark.parametrize("shape,axis", CASES, ids=["x".join(map(str, c[0])) + f"-{c[1]}" for c in CASES])
def test_qdq_flat(hip, oracle_lib, shape, axis, zf32, code):
    rng = np.random.default_rng(int(np.prod(shape)))
    c = 1 if axis is None else shape[axis]
    s = rng.uniform(0.01, 0.2, c).astype(np.float32)
    if c > 2:
        s[1] = 0.0
    x = rng.normal(0, 3, shape).astype(np.float32)
    flat = x.reshape(-1)
    for value in (np.nan, np.inf, -np.inf, -0.0, 1e30, np.float32(2.5) * s[0], np.float32(-3.5) * s[0]):
        flat[rng.integers(0, flat.size)] = value
    zdt = O.F32 if zf32 else code
    z = rng.integers(-3, 4, c).astype(np.float32) if zf32 else (
        rng.integers(0, 100, c).astype(np.uint8) if code != O.I8 else rng.integers(-20, 20, c).astype(np.int8))
    if code in (O.E4M3, O.E5M2) and not zf32:
        z = np.zeros(c, np.uint8)
    view = [1] * len(shape)
    if axis is not None:
        view[axis] = c
    bs, bz = (np.ascontiguousarray(np.broadcast_to(v.reshape(view), shape)) for v in (s, z))
    run = (lambda op, a, din, dout: hip.qdq1(op, a, din, s, z, zdt, dout)) if axis is None else \
        (lambda op, a, din, dout: hip.qdq_axis(op, a, din, s, z, zdt, dout, axis))
    with hip.poisoned():
        q = run("quantize", x, O.F32, code)
    want = oracle_lib.qdq("quantize", x, O.F32, bs, O.F32, bz, zdt, code)
    assert_bitexact(q, want, code, what=f"quantize {shape}")
    with hip.poisoned():
        y = run("dequantize", want, code, O.F32)
    assert_bitexact(y, oracle_lib.qdq("dequantize", want, code, bs, O.F32, bz, zdt, O.F32), O.F32, what=f"dequantize {shape}")
