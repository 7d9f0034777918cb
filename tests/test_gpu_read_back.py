"""Small downloads: sizes around the pinned slots' and a word's, odd addresses,
results of kernels queued just before, long queues, a source in pinned host
memory, an error left by an earlier call, and more threads than slots."""
from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

import hephaestus_amd as hx
from hephaestus_amd import _ffi

from test_gpu_capture import _hip

pytestmark = pytest.mark.gpu

VEC = hx.RocmDenseVectorOps()


@pytest.mark.parametrize("skip,count", [(0, 1), (0, 4), (1, 1), (1, 7), (3, 4093), (0, 4095), (0, 4096), (2, 4096),
                                        (0, 4097), (5, 8000)])
def test_bytes_at_any_address(device, oracle, skip, count):
    host = oracle.uniform_int(2048, seed=count + skip, lo=0, hi=2**32 - 1)
    buffer = device.upload(host)
    out = np.full(count + 2, 0xA5, np.uint8)
    _ffi.check(_ffi.lib().hx_download(device.handle, buffer.ptr + skip, count, out.ctypes.data + 1, count, 1))
    assert np.array_equal(out[1:-1], host.view(np.uint8)[skip:skip + count])
    assert out[0] == 0xA5 and out[-1] == 0xA5


def test_sees_work_queued_before(device):
    a, b = device.upload(np.ones(1 << 20, np.float32)), device.alloc_zeroed(np.float32, 1 << 20)
    dot = VEC.prepare_dot(device, a, a)
    for k in range(1, 40):
        VEC.scale_vector(device, a, 2.0 if k % 2 else 0.5)
        assert VEC.dot_prepared(device, dot, a, a) == (4 if k % 2 else 1) * float(1 << 20)
        VEC.copy_vector(device, a, b)
        assert device.download_owned(b)[-1] == (2.0 if k % 2 else 1.0)


def test_waits_for_long_queued_work(device):
    """Milliseconds of queued work: longer than the host watches the flag."""
    n = 1 << 28
    x, y = device.alloc_zeroed(np.uint32, n), device.alloc_zeroed(np.uint32, n)
    device.write_sub_buffer(x, 0, np.array([7], np.uint32))
    lay = hx.Layout.c_contiguous([n])
    tail = np.zeros(3, np.uint32)
    for k, (src, dst) in enumerate([(x, y), (y, x), (x, y)]):
        for _ in range(4):
            hx.RocmScanOps().scan_axis_into(device, hx.CumSumOp, hx.StridedView(src, lay), 0, hx.ScanDirection.Forward,
                                            hx.StridedView(dst, lay), hx.ScanKind.Inclusive)
        _ffi.check(_ffi.lib().hx_download(device.handle, dst.ptr + 4 * (n - 3), 3, tail.ctypes.data, 3, 4))
        want = np.arange(n - 2, n + 1, dtype=np.uint64)
        want = [7 * np.ones(3, np.uint64), 7 * want, 7 * want * (want + 1) // 2][k]
        assert np.array_equal(tail, want.astype(np.uint32)), k
    x.free()
    y.free()


def test_source_in_pinned_host_memory(device):
    """No slot serves it: the general copy does, as for large downloads."""
    pinned = ctypes.c_void_p()
    assert _hip().hipHostMalloc(ctypes.byref(pinned), ctypes.c_size_t(4096), 0) == 0
    try:
        words = np.frombuffer((ctypes.c_char * 4096).from_address(pinned.value), np.uint32)
        words[:] = np.arange(1024)
        got = np.zeros(100, np.uint32)
        _ffi.check(_ffi.lib().hx_download(device.handle, pinned.value + 40, 100, got.ctypes.data, 100, 4))
        assert np.array_equal(got, np.arange(10, 110))
    finally:
        _hip().hipHostFree(pinned)


def test_an_earlier_error_of_the_thread_is_not_the_downloads(device):
    host = np.arange(5, dtype=np.uint32)
    buffer = device.upload(host)
    assert _hip().hipSetDevice(999) != 0
    try:
        got = device.download_owned(buffer)
    finally:
        _hip().hipGetLastError()
    assert np.array_equal(got, host)


def test_more_threads_than_slots(device):
    buffers = [device.upload(np.arange(17, dtype=np.uint32) + 1000 * t) for t in range(20)]
    right = [0] * len(buffers)

    def work(t):
        for _ in range(100):
            right[t] += np.array_equal(device.download_owned(buffers[t]), np.arange(17, dtype=np.uint32) + 1000 * t)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(len(buffers))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert right == [100] * len(buffers)  # a download that raised ends its thread
