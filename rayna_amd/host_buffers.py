"""Arrays for images in pinned host memory, which the GPU copies to directly.

A copy into ordinary memory goes through the runtime's staging buffer and, for a new array, faults every page in: a 1080p
image's 25 MB take 3.9 ms to a new array, 3.5 to one that is there, and 0.49 into pinned memory (copies alone).  The
memory of an array comes back to a pool when the array and every view of it are gone.  The pool keeps at most
IDLE_BYTES for reuse, the longest unused making room for what comes back.  Arrays larger than that, arrays beyond
PINNED_BYTES in use and arrays for which no pinned memory can be had are ordinary ones.  Any thread may ask for arrays
and drop them.  torch's non-blocking copies of such an array run on after the call: the array may be dropped at once,
but not written to before they end, as with any pinned tensor.

A forked child does not have the parent's pinned memory (the driver keeps it out of forks), so the images alive at a
fork are copied before it, and the child gets the copies as ordinary memory at the same addresses.
"""
from __future__ import annotations

import ctypes as C
import mmap
import os
import sys
import threading
import weakref
from collections import OrderedDict, deque

import numpy as np

IDLE_BYTES = 256 << 20
PINNED_BYTES = 1 << 30
# Waiting for a device that has just worked takes 8-13 us, of the 145 us that a 64x36 frame takes, but one wait does for
# all that was given back before it: so SPARE buffers of up to SPARE_BYTES take turns where torch uses a GPU.
SPARE = 8
SPARE_BYTES = 8 << 20


def _devices_elsewhere_in_use() -> list:
    """The devices on which torch may still be copying from or to dropped arrays: copies from and to pinned memory run on
    after the call when asked not to block."""
    torch = sys.modules.get("torch")
    if torch is None or not hasattr(torch, "cuda") or not torch.cuda.is_initialized():
        return []
    return [d for d in range(torch.cuda.device_count()) if torch._C._cuda_hasPrimaryContext(d)]


def _settle(devices: list) -> bool:
    """Waits for those copies.  False if that cannot be done."""
    from .renderer import lib
    return all(lib().rayna_host_settle(d) == 0 for d in devices)


class _Pool:
    def __init__(self):
        # reentrant: a collection inside a critical section may drop arrays, whose finalizers come back here; they
        # leave their buffers in _returned for later (_busy)
        self._lock = threading.RLock()
        self._busy = False
        self._returned = deque()  # (address, size) given back and not yet counted
        self._idle = OrderedDict()  # address -> (size, the how many-th to be given back), the longest unused first
        self._by_size = {}  # size -> the idle addresses, likewise
        self._given = 0  # buffers given back so far
        self._settled = 0  # no copy is under way in those of them up to here
        self._live = {}  # address -> (bytes asked for, size)
        self._inherited = set()  # in a forked child: the addresses of the parent's arrays
        self._copies = []
        self.idle_bytes = 0
        self.used_bytes = 0

    @staticmethod
    def _size(n: int) -> int:
        """n rounded up to at most an eighth more, so that images of nearly one size share buffers."""
        step = max(4096, 1 << max(0, n.bit_length() - 4))
        return -(-n // step) * step

    def _collect(self) -> list:
        """Makes what was given back idle; the addresses that had to go for it, to be freed."""
        gone = []
        while self._returned:
            address, size = self._returned.popleft()
            if address in self._inherited:  # ordinary memory here, which stays in place
                continue
            del self._live[address]
            self.used_bytes -= size
            self.idle_bytes += size
            self._given += 1
            self._idle[address] = size, self._given
            self._by_size.setdefault(size, deque()).append(address)
            while self.idle_bytes > IDLE_BYTES:
                oldest, (oldest_size, _) = self._idle.popitem(last=False)
                self._by_size[oldest_size].popleft()
                self.idle_bytes -= oldest_size
                gone.append(oldest)
        return gone

    @staticmethod
    def _free(addresses: list):
        if addresses:
            from .renderer import lib
            for a in addresses:
                lib().rayna_host_free(a)

    def take(self, n: int):
        """(address, size) of a buffer of at least n bytes, or None."""
        size = self._size(n)
        got, devices, upto = None, [], 0
        with self._lock:
            if self._busy or size > IDLE_BYTES:
                return None
            self._busy = True
            try:
                gone = self._collect()
                fits = self.used_bytes + size <= PINNED_BYTES
                if fits:
                    self.used_bytes += size
                    same = self._by_size.get(size)
                    if same and self._idle[same[0]][1] <= self._settled:
                        got = same.popleft()
                    elif same:
                        devices = _devices_elsewhere_in_use()
                        if not devices:
                            got = same.pop()
                        elif len(same) >= SPARE or size > SPARE_BYTES:
                            got, upto = same.popleft(), self._given
                    if got is not None:
                        del self._idle[got]
                        self.idle_bytes -= size
                        self._live[got] = n, size
            finally:
                self._busy = False
        self._free(gone)
        if got is not None:
            if upto:
                if not _settle(devices):
                    self.give_back(got, size)
                    return None
                with self._lock:
                    self._settled = max(self._settled, upto)
            return got, size
        if not fits:
            return None
        from .renderer import lib
        p = C.c_void_p()
        if lib().rayna_host_alloc(size, C.byref(p)) != 0:
            with self._lock:
                self.used_bytes -= size
            return None
        with self._lock:
            self._live[p.value] = n, size
        return p.value, size

    def give_back(self, address: int, size: int):
        self._returned.append((address, size))
        with self._lock:
            if self._busy:
                return
            self._busy = True
            try:
                gone = self._collect()
            finally:
                self._busy = False
        self._free(gone)

    def before_fork(self):
        self._lock.acquire()
        self._copies = []
        self._copies = [(a, size, C.string_at(a, n)) for a, (n, size) in self._live.items()]

    def after_fork_in_parent(self):
        self._copies = []
        self._lock.release()

    def after_fork_in_child(self):
        copies, inherited = self._copies, self._inherited
        self.__init__()
        self._inherited = inherited
        libc = C.CDLL(None)
        libc.mmap.restype = C.c_void_p
        libc.mmap.argtypes = [C.c_void_p, C.c_size_t, C.c_int, C.c_int, C.c_int, C.c_long]
        fixed = 0x10  # MAP_FIXED
        for address, size, data in copies:
            at = libc.mmap(address, size, mmap.PROT_READ | mmap.PROT_WRITE,
                           mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS | fixed, -1, 0)
            if at == address:
                C.memmove(address, data, len(data))
            inherited.add(address)


_pool = _Pool()
os.register_at_fork(before=lambda: _pool.before_fork(), after_in_parent=lambda: _pool.after_fork_in_parent(),
                    after_in_child=lambda: _pool.after_fork_in_child())


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
