"""f32 Gemm with B stored [K, N], and K, N and bases that are no multiple of four floats, on
the tiled kernel: both tile shapes, one and several k slices, a k tail of 1 to 3 elements next
to non-finite neighbours, ragged M and N, every bias mode.  Reference: float64 products
(tensor_ops.c:1167-1228 accumulates in double); assert_close's 1e-5 covers f32 sums of at
most 3000 terms."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_close

pytestmark = pytest.mark.gpu

# M, N, K: K mod 4 = 0 .. 3, one slice and several, the 128x256 tiles
SHAPES = [(1, 1, 1), (33, 5, 3), (70, 130, 1100), (65, 67, 1101), (200, 257, 514), (129, 70, 2999), (100, 64, 66),
          (3000, 3001, 35), (40, 1000, 7), (130, 1023, 61)]


@pytest.mark.parametrize("tb", [0, 1], ids=["kn", "nk"])
@pytest.mark.parametrize("bias", ["none", "col", "row", "2d"])
@pytest.mark.parametrize("M,N,K", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_gemm_layouts(hip, M, N, K, bias, tb):
    rng = np.random.default_rng(M + N + K)
    a = rng.normal(0, 1, (M, K)).astype(np.float32)
    b = rng.normal(0, 1 / np.sqrt(K), (N, K) if tb else (K, N)).astype(np.float32)
    c = {"none": None, "col": rng.normal(0, 1, (N,)), "row": rng.normal(0, 1, (M, 1)), "2d": rng.normal(0, 1, (M, N))}[bias]
    c = None if c is None else c.astype(np.float32)
    with hip.poisoned():
        y = hip.gemm(a, O.F32, b, O.F32, c, O.F32, O.F32, 0.75, 1.5, 0, tb)
    rows = np.arange(M) if M * N < 1 << 20 else np.unique(np.r_[rng.choice(M, 40, replace=False), 0, M - 1])
    bt = b.astype(np.float64).T if tb else b.astype(np.float64)
    ref = 0.75 * (a[rows].astype(np.float64) @ bt)
    if c is not None:
        ref = ref + 1.5 * (c if bias == "col" else c[rows]).astype(np.float64)
    assert_close(y[rows], ref.astype(np.float32), O.F32, what=f"{M}x{N}x{K}")


@pytest.mark.parametrize("tb", [0, 1], ids=["kn", "nk"])
def test_gemm_tail_beside_nonfinite(hip, oracle_lib, tb):
    """A chunk that reaches past K meets the next row's first values: they must not count."""
    M, N, K = 37, 70, 65
    rng = np.random.default_rng(1)
    a = rng.normal(0, 1, (M, K)).astype(np.float32)
    b = rng.normal(0, 1, (N, K) if tb else (K, N)).astype(np.float32)
    a[5, 0], a[20, 1] = np.inf, np.nan
    if tb:
        b[9, 0], b[40, 2] = np.nan, -np.inf
    else:
        b[0, 3], b[K - 1, N - 1] = np.nan, np.inf
    y = hip.gemm(a, O.F32, b, O.F32, None, O.F32, O.F32, 1.0, 0.0, 0, tb)
    ref = oracle_lib.gemm(a, O.F32, b, O.F32, None, O.F32, O.F32, 1.0, 0.0, 0, tb)
    assert_close(y, ref, O.F32, what="tail")
    assert np.array_equal(np.isnan(y), np.isnan(ref))


@pytest.mark.parametrize("tb", [0, 1], ids=["kn", "nk"])
def test_gemm_unaligned_bases(hip, tb):
    """Device operands that start one float past a 16-byte boundary."""
    M, N, K = 50, 90, 300
    rng = np.random.default_rng(2)
    a = rng.normal(0, 1, (M, K)).astype(np.float32)
    b = rng.normal(0, 1, (N, K) if tb else (K, N)).astype(np.float32)
    L = hip.lib
    L.gemm_forward.argtypes = [O.PT] * 4 + [ctypes.c_float, ctypes.c_float, ctypes.c_int, ctypes.c_int]
    held = [hip.dev_from(np.concatenate([np.zeros(1, np.float32), v.reshape(-1)]), O.F32) for v in (a, b)]
    views = [L.tensor_wrap_device(t.contents.data + 4, (ctypes.c_int * 2)(*v.shape), 2, O.F32) for t, v in zip(held, (a, b))]
    y = hip.dev_empty((M, N), O.F32)
    L.tensor_ops_hip_clear_error()
    L.gemm_forward(views[0], views[1], O.PT(), y, 1.0, 0.0, 0, tb)
    assert not hip.last_error(), hip.last_error()
    got = hip.dev_read(y, O.F32)
    for t in views + held + [y]:
        L.free_tensor(t)
    bt = b.astype(np.float64).T if tb else b.astype(np.float64)
    assert_close(got, (a.astype(np.float64) @ bt).astype(np.float32), O.F32, what="unaligned")


@pytest.mark.parametrize("M,N,K", [(2048, 1024, 512), (2047, 1023, 1537), (1025, 2047, 33), (2000, 1100, 383), (1024, 2048, 1030)],
                         ids=lambda v: str(v))
def test_gemm_kn_one_pass(hip, M, N, K):
    """B [K, N] with a 128x64 tile for each CU: one pass in parts of 512 k (one part, a part
    ending with K, a last part of a few elements).  Three f32 roundings of parts on sums of at
    most 1537 terms: assert_close's 1e-5."""
    rng = np.random.default_rng(M + N + K)
    a = rng.normal(0, 1, (M, K)).astype(np.float32)
    b = rng.normal(0, 1 / np.sqrt(K), (K, N)).astype(np.float32)
    c = rng.normal(0, 1, (N,)).astype(np.float32)
    with hip.poisoned():
        y = hip.gemm(a, O.F32, b, O.F32, c, O.F32, O.F32, 0.75, 1.5, 0, 0)
    rows = np.unique(np.r_[rng.choice(M, 60, replace=False), 0, 127, 128, M - 1])
    ref = 0.75 * (a[rows].astype(np.float64) @ b.astype(np.float64)) + 1.5 * c.astype(np.float64)
    assert_close(y[rows], ref.astype(np.float32), O.F32, what=f"{M}x{N}x{K}")
