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


@pytest.mark.parametrize("shape,threads", [((1 << 24, 2, 2), 256), (((1 << 22) + 3, 65, 2), 1024), ((3, 2, (1 << 30) + 5), 256),
                                           ((2, 70, 1 << 28), 1024)], ids=lambda v: str(v))
def test_softmax_columns_in_slices(rec, shape, threads):
    """Along an inner dimension: every column block launched once, within the runtime's
    2^32 work-items per dimension (the recorder refuses more, as the runtime does)."""
    launches, err = rec.softmax(shape, 1, O.F16)
    assert not err, err
    cols = 64 if threads == 256 else 32
    assert all(l.block == threads for l in launches)
    assert sum(l.grid[0] for l in launches) == shape[0] * -(-shape[2] // cols)
