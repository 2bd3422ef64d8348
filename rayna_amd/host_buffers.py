"""Arrays for images in pinned host memory, which the GPU copies to directly.

A copy into ordinary memory goes through the runtime's staging buffer and, for a new array, faults every page in:
450 us for 1 MB, 4.7 ms for a 1080p image's 25 MB, against 27 and 444 us into pinned memory (copies alone).  The
memory of an array comes back to a pool when the array and every view of it are gone.  The pool keeps at most
IDLE_BYTES for reuse and frees the rest; arrays beyond PINNED_BYTES in use, or for which no pinned memory can be had,
are ordinary ones.  Any thread may ask for arrays and drop them.
"""
from __future__ import annotations

import ctypes as C
import threading
import weakref

import numpy as np

IDLE_BYTES = 256 << 20
PINNED_BYTES = 1 << 30


class _Pool:
    def __init__(self):
        # reentrant: a collection inside a critical section may drop arrays, whose finalizers come back here
        self._lock = threading.RLock()
        self._idle = {}  # size -> addresses
        self.idle_bytes = 0
        self.used_bytes = 0

    @staticmethod
    def _size(n: int) -> int:
        """n rounded up to at most an eighth more, so that images of nearly one size share buffers."""
        step = max(4096, 1 << max(0, n.bit_length() - 4))
        return -(-n // step) * step

    def take(self, n: int):
        """(address, size) of a buffer of at least n bytes, or None."""
        size = self._size(n)
        with self._lock:
            if self.used_bytes + size > PINNED_BYTES:
                return None
            self.used_bytes += size
            if self._idle.get(size):
                self.idle_bytes -= size
                return self._idle[size].pop(), size
        from .renderer import lib
        p = C.c_void_p()
        if lib().rayna_host_alloc(size, C.byref(p)) != 0:
            with self._lock:
                self.used_bytes -= size
            return None
        return p.value, size

    def give_back(self, address: int, size: int):
        with self._lock:
            self.used_bytes -= size
            if self.idle_bytes + size <= IDLE_BYTES:
                self.idle_bytes += size
                self._idle.setdefault(size, []).append(address)
                return
        from .renderer import lib
        lib().rayna_host_free(address)


_pool = _Pool()


def empty(count: int, dtype) -> np.ndarray:
    """A one-dimensional array of `count` elements, its contents unspecified."""
    n = count * np.dtype(dtype).itemsize
    got = _pool.take(n) if n > 0 else None
    if got is None:
        return np.empty(count, dtype)
    address, size = got
    owner = (C.c_uint8 * n).from_address(address)
    weakref.finalize(owner, _pool.give_back, address, size).atexit = False
    return np.frombuffer(owner, dtype)
