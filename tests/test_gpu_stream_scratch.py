"""The scratch a stream keeps: how far it grows, and what runs where it cannot."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from conftest import assert_matvec_close, bits_equal
from flatrun_amd import _lib, device, synth
from oracle import gguf_np as G

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def test_growth_is_bounded(frq):
    """Batches that need 592, 664 and 448 MiB one after the other: the stream
    holds 1 GiB, where doubling the first capacity would make it 1.7 in all."""
    def free_bytes():                                 # (hipMemGetInfo of the runtime that the library is linked to)
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert frq.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    shapes = [(256, k, 1024) for k in (131072, 147456, 98304)]
    need = [device.batch_plan("Q4_K", *s)[3] for s in shapes]
    assert 512 * MIB < need[0] < need[1] < 700 * MIB and need[2] < 512 * MIB
    kmax = max(k for _, k, _ in shapes)
    w = device.DeviceBuffer.from_host(synth.make_blocks("Q4_K", 256, kmax, seed=1))
    x = device.DeviceBuffer.from_host(np.ones((1024, kmax), np.float32))
    y = device.DeviceBuffer(4 * 256 * 1024)
    s = device.Stream()
    free = free_bytes()
    try:
        for n, k, m in shapes:
            device.gemv("Q4_K", w, x, y, n, k, batch=m, stream=s, w_bytes=synth.nbytes("Q4_K", n, k))
            s.synchronize()
        held = free - free_bytes()
        assert held <= (1024 + 64) * MIB, held // MIB
    finally:
        s.destroy()
        for b in (w, x, y):
            b.free()


@pytest.mark.parametrize("q,n,k,rows", [("Q5_K", 300, 2048, 9), ("Q5_K", 8192, 4096, 16), ("Q1_0", 8192, 4096, 33)])
def test_capture_without_scratch_takes_a_gemv_per_row(frq, q, n, k, rows):
    """A batch of the pair GEMM captured on a stream that has no scratch yet: the
    graph holds one GEMV per row, alone and as a group, and replays their bits;
    outside the capture the same stream takes the pair GEMM."""
    assert device.batch_plan(q, n, k, rows)[0] in ("few", "pair")
    raw, xs = synth.make_blocks(q, n, k, seed=n), synth.make_x(k, seed=rows, batch=rows)
    w, x = device.DeviceBuffer.from_host(raw), device.DeviceBuffer.from_host(xs)
    y, y2, ref = (device.DeviceBuffer(4 * n * rows) for _ in range(3))
    s = device.Stream()
    try:
        for r in range(rows):
            device.gemv(q, w, x.ptr + 4 * k * r, ref.ptr + 4 * n * r, n, k, w_bytes=raw.nbytes)
        device.synchronize()
        with device.Graph.capture(s) as cap:
            device.gemv(q, w, x, y, n, k, batch=rows, stream=s)
            device.gemv_group([(q, w, n, y2, raw.nbytes)], x, k, batch=rows, stream=s)
        want = ref.to_host(np.float32)
        nan = np.full(n * rows, np.nan, np.float32)
        try:
            for _ in range(3):
                for b in (y, y2):
                    _lib.check(_lib.lib().frq_memcpy_h2d(b.ptr, nan.ctypes.data, nan.nbytes))
                cap.launch(s)
                s.synchronize()
                assert bits_equal(y.to_host(np.float32), want) and bits_equal(y2.to_host(np.float32), want)
                device.gemv(q, w, x, y, n, k, batch=rows, stream=s)
                s.synchronize()
                got = y.to_host(np.float32).reshape(rows, n)
                y64, a64 = G.matmul_f64(q, xs[-1], raw, n, k), G.abs_matmul_f64(q, xs[-1], raw, n, k)
                assert_matvec_close(got[-1], y64, a64)
        finally:
            cap.destroy()
    finally:
        for b in (w, x, y, y2, ref):
            b.free()
        s.destroy()
