"""The library's host code without a GPU: load() binds libfirtez_gpu.so to the
stand-in runtime of hip_double.c in this process (one that has loaded no
other HIP runtime: the tests start a fresh interpreter for each case)."""
import ctypes
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))


class Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint32), ("y", ctypes.c_uint32), ("z", ctypes.c_uint32)]


LAUNCH = ctypes.CFUNCTYPE(None, ctypes.c_char_p, Dim3, Dim3, ctypes.c_size_t, ctypes.POINTER(ctypes.c_void_p))


class Launch:
    """A kernel launch: mangled name, grid, block, dynamic LDS and the first
    arguments, each as `size` raw bytes."""

    def __init__(self, name, grid, block, shmem, args):
        self.name, self.grid, self.block, self.shmem = name.decode(), grid.x, block.x, shmem
        self.gridyz, self._args = (grid.y, grid.z), args

    def arg(self, i, ctype):
        return ctype.from_buffer_copy(ctypes.string_at(self._args[i], ctypes.sizeof(ctype)))


class Double:
    def __init__(self, lib, gpu):
        self.lib, self.gpu = lib, gpu
        self.watch = {}
        self.seen = []
        lib.double_held.restype = ctypes.c_size_t
        lib.double_size.restype, lib.double_size.argtypes = ctypes.c_size_t, [ctypes.c_void_p]
        lib.double_mallocs.restype = ctypes.c_long
        lib.double_fail_after.argtypes = [ctypes.c_long]
        lib.double_budget.argtypes = [ctypes.c_size_t]
        lib.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
        lib.hipFree.argtypes = [ctypes.c_void_p]
        self._cb = LAUNCH(self._launch)
        lib.double_on_launch(self._cb)

    def _launch(self, *a):
        x = Launch(*a)
        for key, fn in self.watch.items():
            if key in x.name:
                self.seen.append(fn(x))

    def malloc(self, n):
        p = ctypes.c_void_p()
        assert self.lib.hipMalloc(ctypes.byref(p), n) == 0, "budget"
        return p.value

    def free(self, p):
        assert self.lib.hipFree(p) == 0


def load():
    so = os.path.join(tempfile.mkdtemp(), "libhipdouble.so")
    subprocess.run(["gcc", "-O1", "-w", "-shared", "-fPIC", os.path.join(HERE, "hip_double.c"), "-o", so], check=True)
    lib = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)
    assert "torch" not in sys.modules
    sys.modules["torch"] = None        # its bundled HIP runtime stays out of this process
    from firtez_dz_amd import gpu
    return Double(lib, gpu)
