"""Column-major matrices in the library's device memory, and the HIP runtime the library uses.
(Importing torch here would load a second HIP runtime beside it, whose streams it cannot use.)"""
import ctypes

import numpy as np


class Matrix:
    """A copy of the 2-D array `a` on the device, leading dimension its number of rows."""

    def __init__(self, gb, a):
        self.lib = gb.library()
        self.like = np.asfortranarray(a)
        self.ptr = self.lib.gpublas_dev_alloc(self.like.nbytes)
        assert self.ptr
        self.put(self.like)

    def put(self, a):
        a = np.asfortranarray(a, dtype=self.like.dtype)
        assert self.lib.gpublas_dev_h2d(ctypes.c_void_p(self.ptr), ctypes.c_void_p(a.ctypes.data),
                                        ctypes.c_size_t(a.nbytes), None) == 0
        assert self.lib.gpublas_dev_sync(None) == 0

    def get(self):
        out = np.empty_like(self.like)
        assert self.lib.gpublas_dev_sync(None) == 0
        assert self.lib.gpublas_dev_d2h(ctypes.c_void_p(out.ctypes.data), ctypes.c_void_p(self.ptr),
                                        ctypes.c_size_t(out.nbytes), None) == 0
        assert self.lib.gpublas_dev_sync(None) == 0
        return out

    def free(self):
        self.lib.gpublas_dev_release(ctypes.c_void_p(self.ptr))
