"""Holds the card's free memory, so that the engine's allocations fail as they
do beside other programs.  Kernels that need scratch registers run once on an
engine's queue before (the runtime allocates their scratch then)."""
import contextlib
import ctypes


@contextlib.contextmanager
def device_memory_held(lib, left):
    """All of it but ``left`` bytes and less than as much again: an allocation
    of ``left`` succeeds, one of twice as much fails."""
    lib.hipMalloc.restype = lib.hipFree.restype = ctypes.c_int
    held, spare, size = [], ctypes.c_void_p(), left << 12
    try:
        assert lib.hipMalloc(ctypes.byref(spare), ctypes.c_size_t(left)) == 0
        while size >= left:
            p = ctypes.c_void_p()
            if lib.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0:
                held.append(p)
            else:
                lib.hipGetLastError()
                size //= 2
        lib.hipFree(spare)
        yield
    finally:
        for p in held:
            lib.hipFree(p)
