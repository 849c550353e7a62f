"""Device memory of the current device, by the HIP runtime that the library itself uses."""
import ctypes as C

import narvalengine_amd

MIB = 1 << 20


def _hip():
    narvalengine_amd.lib()  # loads its runtime
    return C.CDLL("libamdhip64.so.7")


def free_bytes() -> int:
    free, total = C.c_size_t(), C.c_size_t()
    assert _hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


class FullCard:
    """Takes the device's memory, untouched, until `leave` bytes at least, and at
    most 256 MiB more, can be allocated beside it (what the runtime says is free
    may be less than that)."""

    def __init__(self, leave: int):
        self.blocks = []
        big = free_bytes() - leave - (4 << 30)
        assert big > 0 and self._take(big)
        while self._take(256 * MIB):
            pass
        for _ in range((leave + 256 * MIB - 1) // (256 * MIB)):
            assert _hip().hipFree(self.blocks.pop()) == 0

    def _take(self, size: int) -> bool:
        p = C.c_void_p()
        if _hip().hipMalloc(C.byref(p), C.c_size_t(size)) != 0:
            _hip().hipGetLastError()  # or the next launch reports it
            return False
        self.blocks.append(p)
        return True

    def free(self):
        for p in self.blocks:
            assert _hip().hipFree(p) == 0
        self.blocks = []
