"""Softmax kernels by row shape against the oracle (tensor_ops.c:1231-1270): a wave or 16
lanes per row, a block of 256 or 1024 threads per row, and 32 or 64 columns per block along
an inner dimension, at the edges of their ranges; rows of -inf, NaN and +inf.  The tolerance
is helpers.assert_close's: 1e-5 relative for f32 (sm_exp's fp32 core is good to 1e-7), one
unit in the last place for f16."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_bitexact, assert_close

pytestmark = pytest.mark.gpu

ROWS = [(5, 1), (17, 16), (33, 17), (16, 32), (7, 33), (6, 64), (9, 65), (3, 256), (2, 257), (1025, 257), (1027, 321),
        (1024, 512), (1024, 513), (512, 1000), (511, 1000), (513, 1025), (512, 2048), (1024, 2049), (1023, 2049)]
# outer, length, inner
COLS = [(3, 1, 5), (2, 1, 257), (5, 2, 256), (3, 2, 300), (4, 3, 65), (2, 8, 63), (2, 9, 65), (1, 33, 64), (4, 64, 7), (2, 65, 33), (1, 128, 31), (1, 257, 32), (2, 512, 3),
        (1, 513, 40)]


def _input(shape, npdt, axis):
    rng = np.random.default_rng(int(np.prod(shape)))
    x = rng.normal(0, 3, shape).astype(npdt)
    rows = np.moveaxis(x, axis, -1)
    n = int(np.prod(rows.shape[:-1]))
    at = np.unravel_index(np.arange(n), rows.shape[:-1])
    if n > 3 and shape[axis] > 1:
        rows[tuple(a[0] for a in at)] = -np.inf               # keeps the start of the maximum: 0 / 0
        rows[tuple(a[1] for a in at) + (0,)] = np.nan
        rows[tuple(a[2] for a in at) + (shape[axis] - 1,)] = np.inf
        rows[tuple(a[3] for a in at) + (0,)] = -np.inf        # one -inf among finite values: 0
    return x


@pytest.mark.parametrize("npdt,dt", [("float32", O.F32), ("float16", O.F16)], ids=["f32", "f16"])
@pytest.mark.parametrize("shape,axis", [(s, 1) for s in ROWS] + [(s, 1) for s in COLS],
                         ids=["x".join(map(str, s)) for s in ROWS + COLS])
def test_softmax_shapes(hip, oracle_lib, shape, axis, npdt, dt):
    x = _input(shape, npdt, axis)
    with hip.poisoned():
        y = hip.softmax(x, dt, dt, axis)
    assert_close(y, oracle_lib.softmax(x, dt, dt, axis), dt, what=f"softmax {shape}")


@pytest.mark.parametrize("shape,din,dout", [((70, 40), O.F64, O.F64), ((600, 700), O.F32, O.F64), ((9, 30), O.F16, O.F32),
                                            ((3, 70, 9), O.F64, O.F32)])
def test_softmax_other_dtypes(hip, oracle_lib, shape, din, dout):
    npdt = {O.F64: "float64", O.F32: "float32", O.F16: "float16"}[din]
    x = _input(shape, npdt, 1)
    assert_close(hip.softmax(x, din, dout, 1), oracle_lib.softmax(x, din, dout, 1), dout, what=f"softmax {shape}")


@pytest.mark.parametrize("M,N", [(5, 30), (33, 200), (1030, 300), (520, 1000)])
def test_gemm_softmax_same_rows(hip, M, N):
    """The split reduction's softmax runs the row kernels above over the slices: the bits of
    the two calls."""
    from tests.test_gpu_qconv import _Dev, _bind
    L = hip.lib
    _bind(L)
    L.gemm_forward.argtypes = [O.PT] * 4 + [ctypes.c_float, ctypes.c_float, ctypes.c_int, ctypes.c_int]
    L.gemm_softmax_forward.argtypes = [O.PT] * 5 + [ctypes.c_float, ctypes.c_float, ctypes.c_int, ctypes.c_int]
    L.softmax_forward.argtypes = [O.PT, O.PT, ctypes.c_int]
    rng = np.random.default_rng(M)
    dev = _Dev(hip)
    try:
        a = dev.put(rng.normal(0, 1, (M, 512)).astype(np.float32), O.F32)
        b = dev.put(rng.normal(0, 0.2, (N, 512)).astype(np.float32), O.F32)
        c = dev.put(rng.normal(0, 1, (N,)).astype(np.float32), O.F32)
        y1, p1, y2, p2 = (dev.empty((M, N), O.F32) for _ in range(4))
        L.tensor_ops_hip_clear_error()
        L.gemm_forward(a, b, c, y1, 1.0, 1.0, 0, 1)
        L.softmax_forward(y1, p1, 1)
        L.gemm_softmax_forward(a, b, c, y2, p2, 1.0, 1.0, 0, 1)
        assert not hip.last_error(), hip.last_error()
        assert_bitexact(hip.dev_read(y2, O.F32), hip.dev_read(y1, O.F32), O.F32, what="logits")
        assert_bitexact(hip.dev_read(p2, O.F32), hip.dev_read(p1, O.F32), O.F32, what="probabilities")
    finally:
        dev.free()


@pytest.mark.parametrize("shape,dtype", [((1 << 24, 2, 2), "float32"), (((1 << 22) + 3, 65, 1, 2), "float16"),
                                         ((1, 2, (1 << 30) + 5), "float16"),
                                         ((1, 3, (1 << 29) + 5), "float16")], ids=["outer24", "outer22", "inner30", "inner29"])
def test_softmax_columns_in_slices(hip, shape, dtype):
    """More column blocks than one launch holds, by the outer or the inner dimension: every
    value against torch's float32 softmax (1e-6 for f32 outputs of at most 1; one unit in the
    last place of f16, 2^-11 of values of at most 1)."""
    import torch
    from tests.test_gpu_qconv import _bind
    L = hip.lib
    _bind(L)
    L.softmax_forward.argtypes = [O.PT, O.PT, ctypes.c_int]
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    x = torch.empty(shape, dtype=getattr(torch, dtype), device="cuda").normal_(0, 2, generator=g)
    y = torch.full_like(x, float("nan"))
    ts = [L.tensor_wrap_device(ctypes.c_void_p(t.data_ptr()), (ctypes.c_int * len(shape))(*shape), len(shape),
                               O.F32 if dtype == "float32" else O.F16) for t in (x, y)]
    torch.cuda.synchronize()
    L.tensor_ops_hip_clear_error()
    L.softmax_forward(*ts, 1)
    assert not hip.last_error(), hip.last_error()
    hip.lib.tensor_ops_hip_sync()
    for t in ts:
        L.free_tensor(t)
    # in pieces along the longest dimension
    dim = int(np.argmax(shape))
    step = 1 << 22 if shape[1] > 2 else 1 << 24
    for a in range(0, shape[dim], step):
        n = min(step, shape[dim] - a)
        want = torch.softmax(x.narrow(dim, a, n).float(), 1)
        d = (y.narrow(dim, a, n).float() - want).abs().max().item()
        assert d <= (1e-6 if dtype == "float32" else 2.0 ** -11), (a, d)
    del x, y
    torch.cuda.empty_cache()
