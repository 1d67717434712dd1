"""The few HIP runtime calls that tests make on their own, through the runtime
that the library loads (torch brings another one: importing it first or last
changes which of them the library gets)."""
import ctypes as C

import numpy as np

_lib = C.CDLL("libamdhip64.so")
_lib.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
_lib.hipFree.argtypes = [C.c_void_p]


def free_bytes():
    """Free device memory once the device is idle."""
    f, t = C.c_size_t(), C.c_size_t()
    assert _lib.hipDeviceSynchronize() == 0
    assert _lib.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


class Buffer:
    """Device memory holding a host array's values."""

    def __init__(self, a):
        self.a, p = np.ascontiguousarray(a), C.c_void_p()
        assert _lib.hipMalloc(C.byref(p), C.c_size_t(self.a.nbytes)) == 0
        self.p = p.value
        assert _lib.hipMemcpy(self.p, self.a.ctypes.data, self.a.nbytes, 1) == 0

    def unchanged(self):
        out = np.empty_like(self.a)
        assert _lib.hipDeviceSynchronize() == 0
        assert _lib.hipMemcpy(out.ctypes.data, self.p, out.nbytes, 2) == 0
        return out.tobytes() == self.a.tobytes()

    def free(self):
        assert _lib.hipFree(self.p) == 0
