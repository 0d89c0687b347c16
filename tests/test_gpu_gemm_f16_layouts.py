"""float16 Gemm in the layouts and sizes that go through chunked copies of the operands (K of
at least 128) and in the small ones below that: every transposition, K around the 8-element
chunks and the 64-k tiles, M and N around the tiles, each tile shape with several k-tiles, one
and several k slices, every bias mode, f16 and f32 outputs.  Products of halves are
exact in f32 and the sums f32 (tensor_ops.c:1167-1228 sums in double): assert_close's one unit
in the last place for f16, 1e-5 for f32."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_close

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 98, 261), (65, 63, 64), (87, 421, 900), (129, 128, 72), (64, 65, 7), (300, 200, 1003), (128, 4100, 40)]
BIAS = {"none": lambda m, n: None, "one": lambda m, n: (1,), "col": lambda m, n: (n,), "row": lambda m, n: (m, 1)}


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("bias", list(BIAS))
@pytest.mark.parametrize("M,N,K", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_gemm_f16_layouts(hip, M, N, K, bias, ta, tb):
    rng = np.random.default_rng(M + N + K)
    a = rng.normal(0, 1, (K, M) if ta else (M, K)).astype(np.float16)
    b = rng.normal(0, 1 / np.sqrt(K), (N, K) if tb else (K, N)).astype(np.float16)
    shape = BIAS[bias](M, N)
    c = None if shape is None else rng.normal(0, 1, shape).astype(np.float32)
    ref = 0.75 * ((a.T if ta else a).astype(np.float64) @ (b.T if tb else b).astype(np.float64))
    ref = ref + (0 if c is None else 1.5 * c.astype(np.float64))
    for ydt in ("float16", "float32"):
        with hip.poisoned():
            y = hip.gemm(a.view(np.uint16), O.F16, b.view(np.uint16), O.F16, c, O.F32, ydt, 0.75, 1.5, ta, tb)
        if ydt == "float16":
            assert_close(y, O.oracle().encode_f32(ref.astype(np.float32), O.F16), O.F16, what="f16")
        else:
            assert_close(y, ref.astype(np.float32), O.F32, what="f32")


@pytest.mark.parametrize("M,N,K", [(1, 64, 128), (8, 1000, 4096), (65, 130, 136), (300, 200, 1000), (129, 2100, 512)],
                         ids=lambda v: str(v))
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_f16_operands_read_in_place(hip, M, N, K, ta, tb):
    """K a multiple of eight: an operand with k along its rows is read where it lies, the
    other from its copy, with one k slice and with several; the bias added once."""
    rng = np.random.default_rng(M * N + K)
    a = rng.normal(0, 1, (K, M) if ta else (M, K)).astype(np.float16)
    b = rng.normal(0, 1 / np.sqrt(K), (N, K) if tb else (K, N)).astype(np.float16)
    c = rng.normal(0, 1, (N,)).astype(np.float32)
    ref = (a.T if ta else a).astype(np.float64) @ (b.T if tb else b).astype(np.float64) + c
    for ydt in ("float16", "float32"):
        with hip.poisoned():
            y = hip.gemm(a.view(np.uint16), O.F16, b.view(np.uint16), O.F16, c, O.F32, ydt, 1.0, 1.0, ta, tb)
        if ydt == "float16":
            assert_close(y, O.oracle().encode_f32(ref.astype(np.float32), O.F16), O.F16, what="f16")
        else:
            assert_close(y, ref.astype(np.float32), O.F32, what="f32")


# M, N, K: 64x128 tiles with 3 (a wrap of its three slots), 4 and 5 k-tiles, 128x128 tiles
# with 2 and 3
TILES = [(1500, 3000, 136), (1030, 4100, 200), (1030, 4100, 320), (2050, 4100, 128), (2050, 4100, 136)]


@pytest.mark.parametrize("M,N,K", TILES, ids=["x".join(map(str, s)) for s in TILES])
@pytest.mark.parametrize("ta", [0, 1])
def test_gemm_f16_larger_tiles(hip, M, N, K, ta):
    """The 64x128 and 128x128 tiles with the Gemm's epilogue, B stored [K, N]."""
    rng = np.random.default_rng(K)
    a = rng.normal(0, 1, (K, M) if ta else (M, K)).astype(np.float16)
    b = rng.normal(0, 1 / np.sqrt(K), (K, N)).astype(np.float16)
    c = rng.normal(0, 1, (N,)).astype(np.float32)
    ref = 0.75 * ((a.T if ta else a).astype(np.float64) @ b.astype(np.float64)) + 1.5 * c.astype(np.float64)
    for ydt in ("float16", "float32"):
        with hip.poisoned():
            y = hip.gemm(a.view(np.uint16), O.F16, b.view(np.uint16), O.F16, c, O.F32, ydt, 0.75, 1.5, ta, 0)
        if ydt == "float16":
            assert_close(y, O.oracle().encode_f32(ref.astype(np.float32), O.F16), O.F16, what="f16")
        else:
            assert_close(y, ref.astype(np.float32), O.F32, what="f32")
