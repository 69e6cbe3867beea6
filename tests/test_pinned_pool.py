"""The page-locked buffers that host calls go through: how many are kept and for
how long (no GPU: the buffers are stand-ins)."""

from __future__ import annotations

import gc
import threading

import flatrun_amd
from flatrun_amd import FrqDeviceError, NativeBackend, device


class Buffer:
    alive = 0

    def __init__(self, nbytes):
        Buffer.alive += 1

    def __del__(self):
        Buffer.alive -= 1


def test_at_most_two_are_kept_and_none_without_a_backend(monkeypatch):
    monkeypatch.setattr(device, "PinnedBuffer", Buffer)
    gc.collect()                                          # backends of other tests
    pool = flatrun_amd._PinnedPool()
    monkeypatch.setattr(flatrun_amd, "_pinned", pool)
    a, b = NativeBackend(), NativeBackend()
    start = threading.Barrier(8)

    def call():
        start.wait()
        for _ in range(50):
            pool.give(pool.take())

    threads = [threading.Thread(target=call) for _ in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    held = [pool.take() for _ in range(5)]
    assert len(set(map(id, held))) == 5 and Buffer.alive == 5
    while held:
        pool.give(held.pop())
    assert Buffer.alive == 2
    del a
    gc.collect()
    assert Buffer.alive == 2
    late = pool.take()
    del b
    gc.collect()
    assert Buffer.alive == 1                              # the one a call still holds
    pool.give(late)
    del late
    assert Buffer.alive == 0


def test_no_memory(monkeypatch):
    def fail(nbytes):
        raise FrqDeviceError(6, "out of memory")

    monkeypatch.setattr(device, "PinnedBuffer", fail)
    pool = flatrun_amd._PinnedPool()
    assert pool.take() is None
    pool.give(None)
