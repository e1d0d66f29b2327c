"""Device memory taken away for a test, through the HIP runtime that
libcolore_amd.so itself has loaded (torch may bring another one)."""
import contextlib
import ctypes

from colore_amd import lib


def free_bytes():
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib.load_amd().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value


@contextlib.contextmanager
def only(room, slack=1 << 26):
    """Leaves about `room` bytes of the device free."""
    amd = lib.load_amd()
    held = []
    try:
        for _ in range(4):   # (the first large block can leave more free than asked for)
            extra = free_bytes() - room
            if extra > slack:
                p = ctypes.c_void_p()
                assert amd.hipMalloc(ctypes.byref(p), ctypes.c_size_t(extra)) == 0
                held.append(p)
        yield
    finally:
        for p in held:
            assert amd.hipFree(p) == 0
