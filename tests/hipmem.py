"""Device memory of the current device, by the HIP runtime that the library itself uses."""
import ctypes as C

import narvalengine_amd


def _hip():
    narvalengine_amd.lib()  # loads its runtime
    return C.CDLL("libamdhip64.so.7")


def free_bytes() -> int:
    free, total = C.c_size_t(), C.c_size_t()
    assert _hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


class Block:
    """`size` bytes of device memory, never touched."""

    def __init__(self, size: int):
        self.p = C.c_void_p()
        assert _hip().hipMalloc(C.byref(self.p), C.c_size_t(size)) == 0

    def free(self):
        assert _hip().hipFree(self.p) == 0
