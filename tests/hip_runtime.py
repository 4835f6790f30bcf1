"""The HIP runtime libgamhip is linked against, for tests that need device or
pinned memory on it (torch bundles a runtime of its own)."""
import ctypes as C

import numpy as np

from mage_amd import gamhip


def runtime():
    gamhip.load()
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
    hip.hipFree.argtypes = [C.c_void_p]
    hip.hipHostFree.argtypes = [C.c_void_p]
    return hip


def used():
    """Bytes of device memory in use."""
    free, total = C.c_size_t(), C.c_size_t()
    hip = runtime()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return total.value - free.value


class Buffer:
    """n doubles of device or pinned host memory, filled from x."""

    def __init__(self, kind, x):
        self.hip, self.kind, self.n = runtime(), kind, x.size
        self.p = C.c_void_p()
        if kind == "device":
            assert self.hip.hipMalloc(C.byref(self.p), x.nbytes) == 0
        else:
            assert self.hip.hipHostMalloc(C.byref(self.p), x.nbytes, 0) == 0
        assert self.hip.hipMemcpy(self.p, x.ctypes.data, x.nbytes, 4) == 0   # hipMemcpyDefault

    @property
    def ptr(self):
        return C.cast(self.p, gamhip.DP)

    def numpy(self):
        out = np.empty(self.n)
        assert self.hip.hipMemcpy(out.ctypes.data, self.p, out.nbytes, 4) == 0
        return out

    def close(self):
        if self.kind == "device":
            self.hip.hipFree(self.p)
        else:
            self.hip.hipHostFree(self.p)
