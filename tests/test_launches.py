"""Which kernels a call launches, on the CPU: the library's own objects over a HIP runtime that
records launches and runs nothing (tests/launches).  Each test is a call that once ended
otherwise."""
import subprocess
import sys

import pytest

from oracle import oracle as O


@pytest.fixture(scope="module")
def rec():
    from tests.launches.recorder import Recorder
    return Recorder()


def kernels(result):
    launches, err = result
    assert not err, err
    return [l.kernel.split("<")[0] for l in launches]


@pytest.mark.parametrize("h,w", [(0, 8), (8, 0), (0, 0)])
def test_conv_f16_of_no_pixels(rec, h, w):
    """An f16 image of no rows or columns whose padding still gives outputs: the host divides
    by H * W nowhere (in a process of its own: it was a SIGFPE)."""
    code = ("from tests.launches.recorder import Recorder; from oracle import oracle as O; "
            f"r = Recorder().conv((1, 16, {h}, {w}), 20, (3, 3), (2, 2, 2, 2), dt=O.F16); "
            "assert not r[1] and len(r[0]) == 1, r")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stderr[-2000:])


@pytest.mark.parametrize("shape,threads", [((1 << 24, 2, 2), 256), (((1 << 22) + 3, 65, 2), 1024), ((3, 2, (1 << 30) + 5), 256), ((3, 3, (1 << 30) + 5), 256),
                                           ((2, 70, 1 << 28), 1024)], ids=lambda v: str(v))
def test_softmax_columns_in_slices(rec, shape, threads):
    """Along an inner dimension: every column block launched once, within the runtime's
    2^32 work-items per dimension (the recorder refuses more, as the runtime does)."""
    launches, err = rec.softmax(shape, 1, O.F16)
    assert not err, err
    cols = 32 if threads == 1024 else 256 if shape[1] <= 2 else 64
    assert all(l.block == threads for l in launches)
    assert sum(l.grid[0] for l in launches) == shape[0] * -(-shape[2] // cols)


def test_softmax_columns_of_two_values(rec):
    """Every thread has a column: 256 of them per block."""
    for length, cols in ((1, 256), (2, 256), (3, 64)):
        (l,), err = rec.softmax((64, length, 16384), 1)
        assert not err and l.grid[0] == 64 * 16384 // cols and l.block == 256


# f32: direct 1x1, 64x64, 128x256, 64x256 and per-pixel plans, all with slices of k
SPLIT_CONVS = [((1, 1024, 14, 14), 256, (1, 1), 1), ((1, 512, 7, 7), 512, (3, 3), 1), ((8, 256, 28, 28), 128, (3, 3), 2),
               ((2, 250, 30, 30), 64, (3, 3), 1), ((1, 19, 14, 14), 30, (3, 3), 1), ((64, 512, 7, 7), 512, (3, 3), 1)]


@pytest.mark.parametrize("codes", [None, O.U8], ids=["f32", "codes"])
@pytest.mark.parametrize("xs,m,k,s", SPLIT_CONVS, ids=["x".join(map(str, c[0])) for c in SPLIT_CONVS])
def test_conv_split_without_memory(rec, xs, m, k, s, codes):
    """No memory for the slices: the same tiles in one pass, and no error."""
    args = (xs, m, k, (k[0] // 2,) * 4, (s, s))
    with_memory = rec.conv(*args, codes=codes)
    rec.no_memory(True)
    try:
        without = rec.conv(*args, codes=codes)
    finally:
        rec.no_memory(False)
    split = kernels(with_memory)
    assert kernels(without) == ["k_conv_tiled"]
    if split != ["k_conv_tiled"]:
        assert split[0] == "k_conv_tiled" and split[1].startswith("k_conv_splitk_reduce")
    else:
        assert xs[1] == 19        # K below two slices


def test_workspace_paths_without_memory(rec):
    """f16 convolution and Gemm copies, f32 Gemm slices: the path that needs none."""
    rec.no_memory(True)
    try:
        assert kernels(rec.conv((32, 128, 28, 28), 128, (3, 3), (1, 1, 1, 1), dt=O.F16)) == ["k_conv_mfma_f32"]
        assert kernels(rec.gemm(512, 1000, 1024, tb=0, dt=O.F16)) == ["k_gemm_mfma_f16"]
        assert kernels(rec.gemm(8, 4096, 4096, dt=O.F16)) == ["k_gemm_f16_nt"]
        assert kernels(rec.gemm(128, 1000, 1024)) == ["k_gemm_f32_nt"]
    finally:
        rec.no_memory(False)


@pytest.mark.parametrize("m,n,k", [(1000, 1000, 128), (300, 64, 200), (1, 64, 136)])
def test_gemm_f16_in_place_under_capture(rec, m, n, k):
    """Operands read where they lie and one k slice need no workspace: the captured call runs
    the eager call's kernel.  Copies need one: the kernel without them."""
    eager, copies = rec.gemm(m, n, k, dt=O.F16), rec.gemm(m, n, k, tb=0, dt=O.F16)
    rec.capturing(True)
    try:
        assert rec.gemm(m, n, k, dt=O.F16) == eager and kernels(eager) == ["k_convh"]
        assert kernels(copies)[-1] == "k_convh" and kernels(rec.gemm(m, n, k, tb=0, dt=O.F16)) == ["k_gemm_mfma_f16"]
        assert kernels(rec.conv((8, 64, 28, 28), 64, (3, 3), (1, 1, 1, 1), dt=O.F16)) == ["k_conv_mfma_f32"]
    finally:
        rec.capturing(False)


@pytest.mark.parametrize("k", [31, 17])
@pytest.mark.parametrize("dt", [O.F32, O.F16, O.U8], ids=["f32", "f16", "codes"])
def test_depthwise_launch_within_the_work_items(rec, k, dt):
    """Many planes of one pixel under a wide window, few to a block: the depthwise kernel's
    blocks would be past 2^32 work-items; the layer runs all the same."""
    args, codes = (1, (k, k), (k // 2,) * 4), O.U8 if dt == O.U8 else None
    r = rec.conv((1 << 28, 1, 1, 1), *args, dt=dt, codes=codes)
    assert len(kernels(r)) == 1
    few = rec.conv((1 << 10, 1, 1, 1), *args, dt=dt, codes=codes)
    assert kernels(few) == ["k_conv_dw"]


def test_small_result_of_another_device(rec):
    """Results that a kernel here may not reach go through the runtime's copy."""
    assert kernels(rec.to_host((1000,), O.F32, owned=True)) == ["k_result"]
    assert kernels(rec.to_host((1000,), O.F32, device=0)) == ["k_result"]
    assert kernels(rec.to_host((1000,), O.F32, device=1)) == []
    assert kernels(rec.to_host((1000,), O.F32, device=-1)) == []


# x shape, output channels, window, stride, groups; whether the channels-last copies are taken
F16_FEW = [((8, 8, 256, 256), 8, 1, 1, 1, 0), ((8, 16, 256, 256), 8, 1, 1, 1, 0), ((8, 16, 256, 256), 16, 1, 1, 1, 1),
           ((8, 2, 256, 256), 8, 3, 1, 1, 1), ((16, 8, 64, 64), 8, 1, 1, 1, 1), ((16, 256, 28, 28), 256, 1, 1, 32, 0),
           ((8, 16, 256, 256), 16, 1, 2, 1, 0), ((8, 32, 256, 256), 8, 1, 2, 1, 0), ((8, 32, 256, 256), 32, 1, 2, 1, 1), ((8, 16, 256, 256), 16, 1, 4, 1, 1), ((8, 3, 256, 256), 8, 3, 8, 1, 1), ((32, 16, 112, 112), 64, 5, 8, 16, 0),
           ((8, 128, 128, 128), 64, 1, 1, 8, 1), ((8, 64, 128, 128), 64, 1, 1, 8, 0),
           ((1, 2, 2000, 2000), 2, 3, 1, 2, 0), ((32, 64, 56, 56), 64, 3, 1, 1, 1)]


@pytest.mark.parametrize("xs,m,k,s,group,copies", F16_FEW, ids=lambda v: str(v).replace(" ", ""))
def test_conv_f16_few_products(rec, xs, m, k, s, group, copies):
    """f16 layers of few products per output over many pixels: the kernel without copies."""
    names = kernels(rec.conv(xs, m, (k, k), (k // 2,) * 4, (s, s), group=group, dt=O.F16))
    assert names[-1] == ("k_convh" if copies else "k_conv_mfma_f32")


# channels, output channels, window, stride; which kernel f32 and codes take, which f16 takes
DW_STRIDES = [(64, 64, 1, 5, 1, 1), (64, 64, 1, 6, 0, 1), (64, 64, 1, 8, 0, 1), (64, 64, 3, 6, 1, 1), (64, 64, 3, 8, 0, 1),
              (16, 64, 1, 3, 1, 1), (16, 64, 1, 4, 0, 1), (16, 64, 1, 6, 0, 0), (16, 64, 3, 4, 0, 1), (16, 64, 5, 8, 0, 0),
              (8, 64, 7, 4, 0, 1), (8, 64, 3, 4, 0, 1), (64, 64, 5, 8, 1, 1), (4, 64, 3, 2, 1, 1), (4, 64, 3, 3, 0, 0), (64, 64, 16, 16, 1, 1), (16, 64, 3, 2, 1, 1), (16, 256, 3, 1, 1, 1)]


@pytest.mark.parametrize("c,m,k,s,f32,f16", DW_STRIDES, ids=lambda v: str(v))
def test_depthwise_strides(rec, c, m, k, s, f32, f16):
    """Strides well past the window: the gathering kernels, for f32 and its codes alike."""
    for dt, codes, dw in ((O.F32, None, f32), (O.F32, O.I8, f32), (O.F16, None, f16)):
        names = kernels(rec.conv((32, c, 112, 112), m, (k, k), (k // 2,) * 4, (s, s), (1, 1), c, dt=dt, codes=codes))
        assert ("k_conv_dw" in names) == bool(dw), names


# x shape, window, stride, pad; whether the row tiles are taken
POOLS = [((1, 16, 33, 33), 3, 1, 1, 0), ((1, 64, 128, 128), 3, 1, 1, 0), ((4, 64, 64, 64), 3, 1, 1, 1), ((1, 64, 50, 50), 3, 1, 1, 0),
         ((4, 64, 50, 50), 3, 1, 1, 1), ((4, 64, 28, 28), 3, 1, 1, 1), ((1, 64, 100, 100), 2, 1, 0, 0), ((4, 64, 100, 100), 2, 1, 0, 1),
         ((1, 64, 33, 33), 5, 1, 2, 0), ((1, 64, 64, 64), 5, 1, 2, 1), ((1, 16, 7, 7), 5, 1, 2, 1), ((1, 3, 1000, 1000), 3, 1, 1, 1), ((1, 16, 128, 128), 5, 1, 2, 1), ((4, 64, 128, 128), 2, 2, 1, 0),
         ((32, 64, 112, 112), 2, 2, 1, 1), ((4, 64, 33, 33), 3, 2, 0, 0), ((8, 128, 33, 33), 3, 2, 0, 1)]


@pytest.mark.parametrize("xs,k,s,p,tiles", POOLS, ids=lambda v: str(v).replace(" ", ""))
def test_maxpool_few_tiles(rec, xs, k, s, p, tiles):
    """Few tiles of wide planes: a wave per output row."""
    assert kernels(rec.maxpool(xs, k, s, p)) == ["k_maxpool_planes" if tiles else "k_maxpool_rows"]


FEW_ROWS = [(1, 10, 100352, 1), (16, 256, 25088, 1), (32, 1000, 3072, 1), (32, 1000, 4096, 0), (24, 1000, 4096, 1), (24, 1000, 6144, 0),
            (32, 64, 25088, 0), (32, 2048, 9216, 1), (32, 2048, 16384, 0), (32, 4096, 25088, 1), (64, 1000, 512, 1), (64, 1000, 1024, 0),
            (64, 4096, 1024, 1), (48, 4096, 4096, 1), (48, 1000, 2048, 0), (64, 4096, 4096, 0), (64, 100, 764, 1), (65, 1000, 512, 0)]


@pytest.mark.parametrize("m,n,k,rows", FEW_ROWS, ids=lambda v: str(v))
def test_gemm_few_rows(rec, m, n, k, rows):
    """Few rows against few columns and a long k: the tiles with their k split.  The same for
    the weight's codes, which return the same bits."""
    for names in (kernels(rec.gemm(m, n, k)), kernels(rec.woq(m, n, k))):
        assert names[0] == ("k_gemm_rows" if rows else "k_gemm_f32_nt")


def test_gpu_cases_reach_their_kernels(rec):
    """The GPU tests' cases named for a k split, a ring of LDS slots or a tile shape take it."""
    from tests import test_gpu_conv_f16, test_gpu_gemm_f16_layouts, test_gpu_gemm_softmax, test_gpu_maxpool_windows
    slices = [c for c in test_gpu_gemm_softmax.CASES if c[0].startswith("slices")]
    rows = {16: "k_softmax_wave<1, 16,", 30: "k_softmax_wave<2, 16,", 200: "k_softmax_wave<4, 64,", 300: "k_softmax_row<1, 1024,",
            400: "k_softmax_wave<8, 64,", 1000: "k_softmax_row<1, 1024,"}
    for name, m, k, n, *_ in slices:
        (gemm, softmax), err = rec.gemm_softmax(m, n, k)
        want = "k_softmax_row<4, 256," if m == 600 else rows[n]
        assert not err and gemm.kernel.startswith("k_gemm_f32_nt") and softmax.kernel.startswith(want), name
        assert softmax.kernel.endswith("SmSlices>"), name
    assert kernels(rec.gemm(70, 1000, 512)) == ["k_gemm_f32_nt", "k_splitk_reduce"]       # the capture tests' Gemm
    for case in test_gpu_conv_f16.CASES:
        name, xs, m, k, pads, strides, dil, group = case
        if name.startswith(("ring", "tiles")):
            launches, err = rec.conv(xs, m, k, pads, strides, dil, group, dt=O.F16)
            bm, bp = name.split("_")[1].split("x")
            assert not err and launches[-1].kernel.startswith(f"k_convh<{bm}, {bp},"), name
        elif name.startswith("few"):
            assert kernels(rec.conv(xs, m, k, pads, strides, dil, group, dt=O.F16)) == ["k_conv_mfma_f32"], name
    for m, n, k in test_gpu_gemm_f16_layouts.TILES:
        for ta in (0, 1):
            launches, err = rec.gemm(m, n, k, ta, 0, O.F16)
            want = "k_convh<128, 128," if m > 2000 else "k_convh<64, 128,"
            assert not err and launches[-1].kernel.startswith(want), (m, n, k)
    for xs, k, stride, pads in test_gpu_maxpool_windows.TILES:
        assert kernels(rec.maxpool(xs, k, stride, pads[0])) == ["k_maxpool_planes"], xs
