"""NativeBackend matmuls of a resident weight: x and y through page-locked
memory (up to 1 MiB of x, 4 MiB of y) or by plain copies beyond that. The same
kernel runs on the same bytes, so the results are those of the device entry
point bit for bit; sizes lie on both sides of each limit, with results that
are no multiple of 16 bytes, an x at an odd address, and k = 0."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import bits_equal
from flatrun_amd import FrqError, device, synth

pytestmark = pytest.mark.gpu

K = 256


@pytest.mark.parametrize("n,rows", [(1, 1), (3, 1), (1001, 1), (64, 1023), (64, 1024), (64, 1025),
                                    (1 << 20, 1), ((1 << 20) + 1, 1), (1025, 1025), (4099, 3)])
def test_same_bits_as_device_call(backend, n, rows):
    rng = np.random.default_rng(n + rows)
    raw = synth.make_blocks("Q4_K", n, K, n)
    w = backend.upload(raw)
    for _ in range(2):                                    # new inputs through the same buffers
        x = rng.standard_normal((rows, K)).astype(np.float32)
        odd = np.zeros(x.nbytes + 1, np.uint8)
        odd[1:] = x.view(np.uint8).reshape(-1)
        xo = odd[1:].view(np.float32).reshape(rows, K)    # not 4-byte aligned
        xd, yd = device.DeviceBuffer.from_host(x), device.DeviceBuffer(rows * n * 4)
        device.gemv("Q4_K", w, xd, yd, n, K, batch=rows)
        device.synchronize()
        want = yd.to_host(np.float32).reshape(rows, n)
        for a in (x, xo):
            assert bits_equal(backend.matmul_q4k(a, w, n, K), want)
        if rows == 1:
            assert bits_equal(backend.matmul_q4k(x[0], w, n, K), want[0])


def test_empty_k_and_errors_leave_the_buffers_usable(backend):
    w = backend.upload(synth.make_blocks("Q4_K", 5, K, 1))
    empty = backend.upload(np.zeros(0, np.uint8))
    x = np.ones(K, np.float32)
    want = backend.matmul_q4k(x, w, 5, K)
    assert not backend.matmul_q4k(np.zeros((2, 0), np.float32), empty, 7, 0).any()
    with pytest.raises(FrqError):
        backend.matmul_q4k(x, w, 6, K)                    # byte size
    with pytest.raises(FrqError):
        backend.matmul_q4k(np.ones(300, np.float32), w, 5, 300)
    assert bits_equal(backend.matmul_q4k(x, w, 5, K), want)
