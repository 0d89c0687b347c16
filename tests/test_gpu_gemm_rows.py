"""Gemm of few rows (k_gemm_rows): one, two and four 16-row tiles at their edges, K below,
at and past a 64-deep chunk and the waves of a block, N around the 16-column blocks, the bias
modes and output types, int8 / uint8 codes bit for bit with DequantizeLinear -> Gemm, and
scales that are not finite.  Reference: the product in float64 (tensor_ops.c:1167-1228
accumulates in double); tolerance assert_close's 1e-5, for f32 sums of at most 4100 terms."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_close

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 4), (1, 1000, 512), (15, 17, 60), (16, 16, 64), (17, 33, 68), (32, 40, 1028), (33, 48, 1024), (48, 4100, 132),
          (64, 100, 1000), (3, 70, 4100), (48, 4096, 1100),
          (64, 100, 764)]
BIAS = {"none": lambda m, n: None, "one": lambda m, n: (1,), "col": lambda m, n: (n,), "row": lambda m, n: (m, 1),
        "2d": lambda m, n: (m, n)}


@pytest.mark.parametrize("ydt", ["float32", "float16"])
@pytest.mark.parametrize("bias", list(BIAS))
@pytest.mark.parametrize("M,N,K", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_gemm_rows(hip, M, N, K, bias, ydt):
    rng = np.random.default_rng(M + N + K)
    a = rng.normal(0, 1, (M, K)).astype(np.float32)
    b = rng.normal(0, 1 / np.sqrt(K), (N, K)).astype(np.float32)
    shape = BIAS[bias](M, N)
    c = None if shape is None else rng.normal(0, 1, shape).astype(np.float32)
    with hip.poisoned():
        y = hip.gemm(a, O.F32, b, O.F32, c, O.F32, ydt, 0.75, 1.5, 0, 1)
    ref = 0.75 * (a.astype(np.float64) @ b.astype(np.float64).T) + (0 if c is None else 1.5 * c.astype(np.float64))
    if ydt == "float16":
        assert_close(y, O.oracle().encode_f32(ref.astype(np.float32), O.F16), O.F16, what="rows")
    else:
        assert_close(y, ref.astype(np.float32), O.F32, what="rows")


@pytest.mark.parametrize("bdt", ["int8", "uint8"])
@pytest.mark.parametrize("M,N,K", [(1, 20, 4), (8, 100, 260), (17, 33, 1028), (40, 50, 700)])
def test_dequantize_gemm_rows(hip, M, N, K, bdt):
    """The bits of DequantizeLinear -> Gemm, with an infinite and a NaN scale among the rows
    (k past K multiplies a zero by (0 - zero point) * scale only if the kernel lets it)."""
    rng = np.random.default_rng(M + N + K)
    lo, hi = (-128, 128) if bdt == "int8" else (0, 256)
    bq = rng.integers(lo, hi, (N, K)).astype(bdt)
    z = rng.integers(-5, 6, N).astype(bdt) if bdt == "int8" else rng.integers(100, 150, N).astype(bdt)
    s = rng.uniform(0.001, 0.02, N).astype(np.float32)
    s[1], s[2] = np.inf, np.nan
    a = np.abs(rng.normal(0, 1, (M, K))).astype(np.float32) + np.float32(0.1)
    bq[1] = np.maximum(bq[1], z[1] + z.dtype.type(1))         # no 0 * inf of its own
    c = rng.normal(0, 1, (N,)).astype(np.float32)
    got = hip.dq_gemm(a, bq, bdt, s, z, 0, c, "float32")
    bd = hip._run(hip.lib.dequantize_linear_axis_forward, [(bq, bdt), (s, O.F32), (z, bdt)], bq.shape, O.F32,
                  ctypes.c_int(0))
    two = hip.gemm(a, O.F32, bd, O.F32, c, O.F32, O.F32, 1.0, 1.0, 0, 1)
    assert np.array_equal(got.view(np.uint32), two.view(np.uint32))
    assert np.all(got[:, 1] == np.inf) and np.all(np.isnan(got[:, 2]))
    keep = [n for n in range(N) if n not in (1, 2)]
    ref = a.astype(np.float64) @ bd[keep].astype(np.float64).T + c[keep]
    assert_close(got[:, keep], ref.astype(np.float32), O.F32, what="codes")
