"""Holds the card's free memory, so that the engine's allocations fail as they
do beside other programs.  Kernels that need scratch registers run once on an
engine's queue before (the runtime allocates their scratch then)."""
import contextlib
import ctypes


@contextlib.contextmanager
def device_memory_held(lib, left=32 << 20):
    """All but about ``left`` bytes, in blocks down to that size."""
    held, size = [], 64 << 30
    lib.hipMalloc.restype = lib.hipFree.restype = ctypes.c_int
    try:
        while size >= left:
            p = ctypes.c_void_p()
            if lib.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0:
                held.append(p)
            else:
                lib.hipGetLastError()
                size //= 2
        yield
    finally:
        for p in held:
            lib.hipFree(p)
