"""The library's dispatch on the CPU: its objects linked against hip_stub.cpp, whose kernel
launches are recorded instead of run.  Tensors are headers over addresses that nothing reads."""
import collections
import ctypes
import fcntl
import os
import subprocess

from onnx_translator_amd import build as B
from oracle import oracle as O

HERE = os.path.dirname(os.path.abspath(__file__))
OUT = os.path.join(HERE, "_build", "liblaunches.so")
Launch = collections.namedtuple("Launch", "kernel grid block")


def _newer(path, sources):
    return os.path.exists(path) and all(os.path.getmtime(path) >= os.path.getmtime(s) for s in sources)


def build():
    """Links (compiling what is stale) and returns the recording library's path; one process
    at a time."""
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    os.makedirs(B.OBJ, exist_ok=True)
    with open(OUT + ".lock", "w") as lock:
        fcntl.flock(lock, fcntl.LOCK_EX)
        return _build()


def _build():
    headers = [os.path.join(B.CSRC, f) for f in os.listdir(B.CSRC) if f.endswith(".h")]
    stub = os.path.join(HERE, "hip_stub.cpp")
    objs = [os.path.join(B.OBJ, os.path.splitext(s)[0] + ".o") for s in B.SOURCES]
    stale = [s for s, o in zip(B.SOURCES, objs) if not _newer(o, headers + [os.path.join(B.CSRC, s)])]
    with B.cf.ThreadPoolExecutor(max_workers=4) as ex:
        list(ex.map(B._compile, stale))
    if not _newer(OUT, objs + [stub]):
        rocm = os.path.dirname(os.path.dirname(os.path.realpath(B.HIPCC)))
        subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", rocm + "/include",
                        "-Wl,-Bsymbolic", "-o", OUT, stub, *objs, "-lpthread"], check=True)
    return OUT


class Recorder:
    def __init__(self):
        L = self.lib = ctypes.CDLL(build())
        cf, ci, PT = ctypes.c_float, ctypes.c_int, O.PT
        L.stub_launches.restype = ctypes.c_void_p
        L.stub_malloc_limit.argtypes = [ctypes.c_size_t]
        L.tensor_wrap_device.restype = PT
        L.tensor_wrap_device.argtypes = [ctypes.c_void_p, ctypes.POINTER(ci), ci, ci]
        L.free_tensor.argtypes = [PT]
        L.create_tensor_device_empty.restype = PT
        L.create_tensor_device_empty.argtypes = [ctypes.POINTER(ci), ci, ci]
        L.tensor_ops_hip_last_error.restype = ctypes.c_char_p
        L.conv2d_forward.argtypes = [PT] * 4 + [ctypes.POINTER(O.CConvParams)]
        L.conv2d_fused_forward.argtypes = [PT] * 4 + [ci, PT, ctypes.POINTER(O.CConvParams)]
        L.dequantize_conv2d_fused_forward.argtypes = [PT] * 6 + [ci, PT, ctypes.POINTER(O.CConvParams)]
        L.max_pool_forward.argtypes = [PT, PT, ctypes.POINTER(O.CPoolParams)]
        L.gemm_forward.argtypes = [PT] * 4 + [cf, cf, ci, ci]
        L.gemm_softmax_forward.argtypes = [PT] * 5 + [cf, cf, ci, ci]
        L.dequantize_gemm_forward.argtypes = [PT] * 4 + [ci, PT, PT, cf, cf, ci, ci]
        L.softmax_forward.argtypes = [PT, PT, ci]
        self._at = 1 << 40

    def tensor(self, shape, dt, offset=0):
        """A device tensor's header over an address of its own (aligned, plus offset)."""
        t = self.lib.tensor_wrap_device(self._at + offset, (ctypes.c_int * len(shape))(*shape), len(shape), dt)
        self._at += 1 << 36
        return t

    def no_memory(self, on):
        """Device allocations fail from here on (and the pool's cached buffers are given up)."""
        self.lib.stub_malloc_limit(0 if on else (1 << 64) - 1)
        if on:      # an allocation that fails
            assert not self.lib.create_tensor_device_empty(O._ints([1 << 30]), 1, O.F32)

    def capturing(self, on):
        """The stream counts as being captured into a graph."""
        self.lib.stub_capturing(1 if on else 0)

    def to_host(self, shape, dt, owned=False, device=-1):
        """(launches, error) of reading a tensor of the library's own memory, or of memory that
        the runtime says lies on a device (-1: that it does not know)."""
        t = self.lib.create_tensor_device_empty(O._ints(shape), len(shape), dt) if owned else self.tensor(shape, dt)
        self.lib.stub_pointer_device(device)
        try:
            return self.call("tensor_to_host", t, ctypes.create_string_buffer(1 << 16))
        finally:
            self.lib.stub_pointer_device(-1)

    def call(self, fn, *args):
        """(launches, error) of one call of the library's fn."""
        self._take()
        self.lib.tensor_ops_hip_clear_error()
        getattr(self.lib, fn)(*args)
        err = self.lib.tensor_ops_hip_last_error()
        for a in args:
            if isinstance(a, O.PT) and a:
                self.lib.free_tensor(a)
        return self._take(), err.decode() if err else ""

    def _take(self):
        p = self.lib.stub_launches()
        text = ctypes.string_at(p).decode()
        ctypes.CDLL(None).free(ctypes.c_void_p(p))
        out = []
        for line in text.splitlines():
            kernel, grid, block = line.split("|")
            name = kernel.replace("void ", "").replace("tohip::(anonymous namespace)::", "").replace("tohip::", "")
            out.append(Launch(name.split("(")[0], tuple(map(int, grid.split())), int(block)))
        return out

    # ---- one call each, by shapes
    def conv(self, xs, m, k, pads=(0, 0, 0, 0), strides=(1, 1), dil=(1, 1), group=1, dt=O.F32, odt=None, bdt=O.F32, codes=None):
        n, c, h, w = xs
        oh = (h + pads[0] + pads[2] - dil[0] * (k[0] - 1) - 1) // strides[0] + 1
        ow = (w + pads[1] + pads[3] - dil[1] * (k[1] - 1) - 1) // strides[1] + 1
        keep = [O._ints(pads), O._ints(strides), O._ints(dil)]
        p = O.CConvParams()
        p.pads, p.strides, p.dilations = [ctypes.cast(v, ctypes.POINTER(ctypes.c_int)) for v in keep]
        p.group = group
        wt = self.tensor((m, c // group) + tuple(k), O.F32 if codes else dt)
        b = self.tensor((m,), bdt) if bdt is not None else O.PT()
        y = self.tensor((n, m, oh, ow), O.F32 if codes else (dt if odt is None else odt))
        if codes:
            return self.call("dequantize_conv2d_fused_forward", self.tensor(xs, codes), self.tensor((1,), O.F32),
                             self.tensor((1,), codes), wt, b, O.PT(), 0, y, ctypes.byref(p))
        return self.call("conv2d_forward", self.tensor(xs, dt), wt, b, y, ctypes.byref(p))

    def maxpool(self, xs, k, stride, pad):
        n, c, h, w = xs
        out = [(v + 2 * pad - k) // stride + 1 for v in (h, w)]
        keep = [O._ints((pad,) * 4), O._ints((stride,) * 2), O._ints((1, 1)), O._ints((k, k))]
        p = O.CPoolParams()
        p.pads, p.strides, p.dilations, p.kernel_shape = [ctypes.cast(v, ctypes.POINTER(ctypes.c_int)) for v in keep]
        return self.call("max_pool_forward", self.tensor(xs, O.F32), self.tensor([n, c] + out, O.F32), ctypes.byref(p))

    def gemm(self, m, n, k, ta=0, tb=1, dt=O.F32, bias=True):
        a, b = self.tensor((k, m) if ta else (m, k), dt), self.tensor((n, k) if tb else (k, n), dt)
        return self.call("gemm_forward", a, b, self.tensor((n,), O.F32) if bias else O.PT(), self.tensor((m, n), dt),
                         1.0, 1.0, ta, tb)

    def gemm_softmax(self, m, n, k):
        return self.call("gemm_softmax_forward", self.tensor((m, k), O.F32), self.tensor((n, k), O.F32),
                         self.tensor((n,), O.F32), self.tensor((m, n), O.F32), self.tensor((m, n), O.F32), 1.0, 1.0, 0, 1)

    def woq(self, m, n, k):
        return self.call("dequantize_gemm_forward", self.tensor((m, k), O.F32), self.tensor((n, k), O.I8),
                         self.tensor((n,), O.F32), self.tensor((n,), O.I8), 0, self.tensor((n,), O.F32),
                         self.tensor((m, n), O.F32), 1.0, 1.0, 0, 1)

    def softmax(self, shape, axis, dt=O.F32, odt=None):
        return self.call("softmax_forward", self.tensor(shape, dt), self.tensor(shape, dt if odt is None else odt), axis)
