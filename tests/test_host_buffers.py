"""The pool of pinned image buffers: its bounds, reuse and fallbacks on a stand-in allocator, and on the GPU that an
image is never overwritten while it or a view of it is held."""
import ctypes as C
import gc
import mmap
import os
import threading

import numpy as np
import pytest

from rayna_amd import Renderer, host_buffers, presets, renderer
from rayna_amd import _abi as A
from rayna_amd.batch import BatchRenderer, Request


class FakeLib:
    """rayna_host_alloc / rayna_host_free over ordinary memory."""

    def __init__(self, fail=False):
        self.fail, self.held = fail, {}

    def rayna_host_alloc(self, size, out):
        if self.fail:
            return 1
        a = np.zeros(size, np.uint8)
        self.held[a.ctypes.data] = a
        out._obj.value = a.ctypes.data
        return 0

    def rayna_host_free(self, address):
        del self.held[address]


@pytest.fixture
def fake(monkeypatch):
    lib = FakeLib()
    monkeypatch.setattr(renderer, "lib", lambda: lib)
    monkeypatch.setattr(host_buffers, "_pool", host_buffers._Pool())
    return lib


def test_reuse_only_after_the_last_view(fake):
    a = host_buffers.empty(1000, np.float32)
    at = a.ctypes.data
    view = a[10:20].reshape(2, 5)
    del a
    gc.collect()
    b = host_buffers.empty(1000, np.float32)
    assert b.ctypes.data != at and b.flags.writeable and b.shape == (1000,)
    del view
    gc.collect()
    assert host_buffers.empty(990, np.float32).ctypes.data == at


def test_bounds(fake, monkeypatch):
    monkeypatch.setattr(host_buffers, "IDLE_BYTES", 3 * 4096)
    monkeypatch.setattr(host_buffers, "PINNED_BYTES", 5 * 4096)
    arrays = [host_buffers.empty(4096, np.uint8) for _ in range(7)]
    assert len(fake.held) == 5 and host_buffers._pool.used_bytes == 5 * 4096
    del arrays
    gc.collect()
    assert len(fake.held) == 3 and host_buffers._pool.used_bytes == 0


def test_without_pinned_memory_and_empty(fake):
    fake.fail = True
    assert host_buffers.empty(5, np.float32).shape == (5,) and host_buffers._pool.used_bytes == 0
    assert host_buffers.empty(0, np.float32).shape == (0,)


def test_threads(fake):
    bad = []

    def work(k):
        for i in range(300):
            a = host_buffers.empty(1 + (i * 37 + k) % 5000, np.uint8)
            a[:] = k
            b = host_buffers.empty(1 + (i * 53 + k) % 5000, np.uint8)
            b[:] = k + 100
            if not (a == k).all():
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    gc.collect()
    assert not bad and host_buffers._pool.used_bytes == 0


@pytest.mark.gpu
def test_held_images_keep_their_values(gpu):
    frames, copies = [], []
    for seed in range(4):
        sc, cam, opts = presets.cornell(width=65, height=43, samples=2, seed=seed)
        with Renderer(sc, cam, opts) as r:
            for out in (r.render(), r.render_srgb8(), r.render(layout="rowmajor")):
                frames.append(out.img[1:])
                copies.append(out.img[1:].copy())
    for a, b in zip(frames, copies):
        assert np.array_equal(a, b)


@pytest.mark.gpu
def test_failed_pinned_allocation_leaves_no_error_behind(gpu):
    """More bytes than any machine has, refused through the real library: the frames and batches that follow on the
    same thread take no notice, whichever entry point reads the runtime's last error next."""
    sc, cam, opts = presets.cornell(width=33, height=21, samples=2)
    with Renderer(sc, cam, opts) as r, BatchRenderer([sc]) as b:
        ref = r.render(layout="rowmajor").img.copy()
        p = C.c_void_p()
        for _ in range(2):
            assert renderer.lib().rayna_host_alloc(1 << 60, C.byref(p)) == A.RAYNA_OUT_OF_MEMORY and not p.value
            r.clear_accumulation()
            assert np.array_equal(r.render(layout="rowmajor").img, ref)
            assert renderer.lib().rayna_host_alloc(1 << 60, C.byref(p)) == A.RAYNA_OUT_OF_MEMORY
            assert np.array_equal(b.render([Request(0, cam, opts)])[0][0], ref)


def test_allocations_do_not_touch_the_last_creation_error():
    """Any thread may allocate (images do, with the GIL released), so the process-wide text that rayna_last_error(NULL)
    reports for another thread's rayna_create stays as it is, after failures and successes alike."""
    L = renderer.lib()
    out = C.c_void_p()
    assert L.rayna_create(None, None, None, C.byref(out)) == A.RAYNA_INVALID_ARGUMENT
    text = L.rayna_last_error(None)
    assert b"null" in text
    assert L.rayna_host_alloc(0, C.byref(out)) == A.RAYNA_INVALID_ARGUMENT
    assert L.rayna_host_alloc(64, None) == A.RAYNA_INVALID_ARGUMENT
    assert L.rayna_last_error(None) == text
    if L.rayna_host_alloc(4096, C.byref(out)) == A.RAYNA_OK:  # (no device here: refused)
        L.rayna_host_free(out)
    assert L.rayna_last_error(None) == text


def test_a_new_size_takes_the_place_of_one_no_longer_asked_for(fake, monkeypatch):
    """A window resized, a server's mixed requests: after a few images of the new size, no allocation and no free."""
    monkeypatch.setattr(host_buffers, "IDLE_BYTES", 8 * 4096)
    calls = []
    for name in ("rayna_host_alloc", "rayna_host_free"):
        f = getattr(fake, name)
        monkeypatch.setattr(fake, name, lambda *a, f=f, name=name: (calls.append(name), f(*a))[1])
    old = [host_buffers.empty(3 * 4096, np.uint8) for _ in range(2)] + [host_buffers.empty(4096, np.uint8)]
    del old
    gc.collect()
    for n in (2 * 4096, 5 * 4096):
        for k in range(50):
            host_buffers.empty(n, np.uint8)
            gc.collect()
            if k == 2:
                del calls[:]
        assert not calls
    assert host_buffers._pool.idle_bytes <= 8 * 4096
    assert sum(a.size for a in fake.held.values()) == host_buffers._pool.idle_bytes


def test_the_longest_unused_buffer_goes_first(fake, monkeypatch):
    monkeypatch.setattr(host_buffers, "IDLE_BYTES", 3 * 4096)
    a, b, c = (host_buffers.empty(4096, np.uint8) for _ in range(3))
    at = {k: v.ctypes.data for k, v in (("a", a), ("b", b), ("c", c))}
    del b  # each given back here
    del c
    del a
    two = host_buffers.empty(2 * 4096, np.uint8)
    del two
    gc.collect()
    assert at["b"] not in fake.held and at["c"] not in fake.held and at["a"] in fake.held
    assert host_buffers.empty(4096, np.uint8).ctypes.data == at["a"]


def test_images_larger_than_the_pool_keeps_are_ordinary(fake, monkeypatch):
    monkeypatch.setattr(host_buffers, "IDLE_BYTES", 3 * 4096)
    a = host_buffers.empty(4 * 4096, np.uint8)
    assert not fake.held and a.shape == (4 * 4096,) and host_buffers._pool.used_bytes == 0


def _exit_of_forked_child(work):
    """The exit code of a forked child that runs work(), or minus the signal that ended it."""
    pid = os.fork()
    if pid == 0:
        code = 1
        try:
            code = 0 if work() else 2
        finally:
            os._exit(code)
    return os.waitstatus_to_exitcode(os.waitpid(pid, 0)[1])


class ForkLib:
    """rayna_host_alloc / rayna_host_free over memory that a forked child does not have, as pinned memory."""

    def __init__(self):
        self.maps, self.freed = {}, []

    def rayna_host_alloc(self, size, out):
        m = mmap.mmap(-1, size)
        m.madvise(mmap.MADV_DONTFORK)
        out._obj.value = C.addressof(C.c_char.from_buffer(m))
        self.maps[out._obj.value] = m
        return 0

    def rayna_host_free(self, address):
        self.freed.append(address)


def test_forked_children_have_the_images(monkeypatch):
    """A child forked with an image in hand (a worker process that saves it) reads the image's values, in its own
    memory; what the parent does with the buffer later is not seen, and the child gives nothing back."""
    lib = ForkLib()
    monkeypatch.setattr(renderer, "lib", lambda: lib)
    monkeypatch.setattr(host_buffers, "_pool", host_buffers._Pool())
    idle = host_buffers.empty(3000, np.uint8)
    del idle
    gc.collect()
    images = [host_buffers.empty(n, np.float32) for n in (5, 1024, 70001)]
    for k, a in enumerate(images):
        a[:] = np.arange(a.size) + k
    views = [a[1:] for a in images]

    def child():
        ok = all(np.array_equal(views[k], np.arange(1, images[k].size) + k) for k in range(3))
        views[1][3] = 77.0  # writable, and its own
        ok = ok and images[1][4] == 77.0
        new = host_buffers.empty(3000, np.uint8)  # not the idle buffer, which the child does not have
        new[:] = 9
        del images[:], views[:]
        gc.collect()
        return ok and not lib.freed and (new == 9).all()

    del a
    assert _exit_of_forked_child(child) == 0
    assert images[1][4] == 5.0 and host_buffers._pool.used_bytes > 0
    assert host_buffers.empty(3000, np.uint8).size == 3000  # the pool goes on


@pytest.mark.gpu
def test_forked_children_have_rendered_images(gpu):
    sc, cam, opts = presets.cornell(width=65, height=43, samples=2)
    with Renderer(sc, cam, opts) as r:
        img = r.render().img
        copy = img.copy()
        assert _exit_of_forked_child(lambda: np.array_equal(img, copy)) == 0
        r.clear_accumulation()
        assert np.array_equal(r.render().img, copy) and np.array_equal(img, copy)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["global", "thread_local", "relaxed"])
@pytest.mark.parametrize("thread", [False, True])
def test_images_may_be_dropped_while_a_graph_is_captured(gpu, monkeypatch, mode, thread):
    """A collection may come at any time, also between the launches of a capture, on its thread or another: the memory
    that the pool then frees, or hands out again, does not break the capture."""
    import torch
    monkeypatch.setattr(host_buffers, "_pool", host_buffers._Pool())
    monkeypatch.setattr(host_buffers, "IDLE_BYTES", 5 << 20)
    monkeypatch.setattr(host_buffers, "SPARE_BYTES", 0)
    images = [host_buffers.empty(4 << 20, np.uint8) for _ in range(3)]
    x = torch.zeros(64, device="cuda")
    y = torch.zeros(64, device="cuda")
    torch.cuda.synchronize()

    def drop_and_take():
        images.clear()
        images.append(host_buffers.empty(4 << 20, np.uint8))  # one that was kept, once its copies have ended

    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode=mode):
        x.add_(1)
        if thread:
            t = threading.Thread(target=drop_and_take)
            t.start()
            t.join()
        else:
            drop_and_take()
        y.copy_(x)
    assert host_buffers._pool.used_bytes == 4 << 20 and host_buffers._pool.idle_bytes == 0
    for k in range(4):
        g.replay()
        torch.cuda.synchronize()
        assert (y == k + 1).all()
        (x * 2).sum().item()  # the program's own work between replays


@pytest.mark.gpu
@pytest.mark.parametrize("to_device", [True, False])
@pytest.mark.parametrize("side", [False, True])
def test_copies_in_flight_have_ended_before_a_buffer_is_used_again(gpu, monkeypatch, to_device, side):
    """torch copies from and to pinned memory without waiting when asked not to block (with ordinary memory it waits):
    a program that drops a frame after such a copy, while the device is busy, has that frame on the device, and the
    next image keeps what is written to it."""
    import torch
    monkeypatch.setattr(host_buffers, "_pool", host_buffers._Pool())
    monkeypatch.setattr(host_buffers, "SPARE_BYTES", 0)
    a = torch.randn(8192, 8192, device="cuda", dtype=torch.bfloat16)
    dev = torch.full((1 << 18,), 3.0, device="cuda")
    stream = torch.cuda.Stream() if side else torch.cuda.current_stream()
    torch.cuda.synchronize()
    img = host_buffers.empty(1 << 18, np.float32)
    img[:] = 7.0
    at = img.ctypes.data
    with torch.cuda.stream(stream):
        for _ in range(60):  # tens of milliseconds of work before the copy
            b = a @ a
        if to_device:
            dev.copy_(torch.from_numpy(img), non_blocking=True)
        else:
            torch.from_numpy(img).copy_(dev, non_blocking=True)
    del img
    gc.collect()
    new = []
    while not new or new[-1].ctypes.data != at:
        new.append(host_buffers.empty(1 << 18, np.float32))
        new[-1][:] = -1.0
    torch.cuda.synchronize()
    assert (dev == (7.0 if to_device else 3.0)).all() and all((a == -1.0).all() for a in new)
    del b


@pytest.fixture(autouse=True)
def only_this_library_uses_a_device(request, monkeypatch):
    """For the tests on a stand-in library, whatever ran in the process before."""
    if "fake" in request.fixturenames:
        monkeypatch.setattr(host_buffers, "_devices_elsewhere_in_use", lambda: [])


def test_a_buffer_that_may_be_in_use_is_not_handed_out(fake, monkeypatch):
    """Where torch uses a device, a buffer is handed out again after a wait for the device that began after it was given
    back, one wait for all of these; small ones take turns; and where the wait fails, the array is an ordinary one."""
    waits, ok = [], True
    monkeypatch.setattr(host_buffers, "_devices_elsewhere_in_use", lambda: [0, 1])
    monkeypatch.setattr(host_buffers, "_settle", lambda devices: (waits.append(devices), ok)[1])
    monkeypatch.setattr(host_buffers, "SPARE_BYTES", 4096)

    def use(n):
        a = host_buffers.empty(n, np.uint8)
        return a.ctypes.data

    at = [use(1000) for _ in range(100)]
    assert len(fake.held) == len(set(at)) == host_buffers.SPARE
    assert 100 / host_buffers.SPARE - 2 <= len(waits) <= 100 / host_buffers.SPARE and waits[0] == [0, 1]
    del waits[:]
    assert len({use(5000) for _ in range(10)}) == 1 and len(waits) == 9  # larger: a wait each time
    a = host_buffers.empty(5000, np.uint8)
    del a, waits[:]
    ok = False
    b = host_buffers.empty(5000, np.uint8)
    assert len(waits) == 1 and b.ctypes.data not in fake.held and host_buffers._pool.used_bytes == 0
    ok = True
    assert use(5000) in fake.held
