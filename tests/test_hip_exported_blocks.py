"""Exported storage after its release: kept for an allocation of the same size
that waits for all work on the device, bounded, given back, and taken by one
owner at a time."""

from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

from conftest import require_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    require_gpu()
    import tensorcx_hip_capi
    lib = tensorcx_hip_capi.lib()
    lib.tcx_hip_release_uncached.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p]
    lib.tcx_hip_release_uncached.restype = None
    lib.tcx_hip_scalar_op.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64,
                                      ctypes.c_double, ctypes.c_int, ctypes.c_void_p]
    return tensorcx_hip_capi


def allocate(capi, nbytes):
    ptr, owner = ctypes.c_void_p(), ctypes.c_void_p()
    capi.check(capi.lib().tcx_hip_allocate(nbytes, ctypes.byref(ptr), ctypes.byref(owner)), "allocate")
    assert not owner.value
    return ptr


def release(capi, ptr, nbytes):
    capi.lib().tcx_hip_release_uncached(ptr, nbytes, None)


def give_back(capi):
    """Leaving any pool frees the kept blocks."""
    pool = ctypes.c_void_p()
    capi.check(capi.lib().tcx_hip_pool_create(0, 1, None, ctypes.byref(pool)), "pool")
    capi.check(capi.lib().tcx_hip_pool_enter(pool), "enter")
    capi.check(capi.lib().tcx_hip_pool_exit(pool), "exit")
    capi.lib().tcx_hip_pool_destroy(pool)


def other_stream(capi):
    streams = []
    thread = threading.Thread(target=lambda: streams.append(capi.stream()))
    thread.start()
    thread.join()
    return streams[0]


def test_work_queued_before_the_release_finishes_first(capi):
    """Another stream still reads the block when it is released: whoever gets
    it next may write only after that."""
    n = 1 << 22
    stream = other_stream(capi)
    a, b, c = (capi.DeviceArray((2048, 2048)) for _ in range(3))
    for t in (a, b):
        capi.check(capi.lib().tcx_hip_fill(0, t.ptr, 2048 * 2048, 0.0, capi.stream()), "fill")
    copy = capi.DeviceArray((n,))
    for attempt in range(3):
        x = allocate(capi, 4 * n)
        capi.check(capi.lib().tcx_hip_fill(0, x, n, float(attempt + 1), capi.stream()), "fill")
        capi.synchronize()
        for _ in range(30):  # some milliseconds in front of the read
            capi.gemm(a.ptr, b.ptr, c.ptr, capi.gemm_desc(2048, 2048, 2048), stream)
        capi.check(capi.lib().tcx_hip_scalar_op(1, 0, x, copy.ptr, n, 0.0, 0, stream), "copy")
        release(capi, x, 4 * n)
        y = allocate(capi, 4 * n)
        assert y.value == x.value  # kept, and the newest of its size
        capi.check(capi.lib().tcx_hip_fill(0, y, n, -1.0, capi.stream()), "fill")
        capi.synchronize()
        capi.check(capi.lib().tcx_hip_stream_synchronize(stream), "synchronize")
        np.testing.assert_array_equal(copy.numpy(), np.full(n, attempt + 1, np.float32))
        release(capi, y, 4 * n)
    give_back(capi)


def test_bounds_and_giving_back(capi):
    free = lambda: capi.device_info()["free_bytes"]  # noqa: E731
    give_back(capi)
    start, mib = free(), 1 << 20
    blocks = [allocate(capi, 100 * mib) for _ in range(8)]
    for ptr in blocks:
        release(capi, ptr, 100 * mib)
    assert 0 < start - free() <= 520 * mib  # five of the eight are kept
    again = [allocate(capi, 100 * mib) for _ in range(8)]
    assert {p.value for p in again[:5]} == {p.value for p in blocks[3:]}
    for ptr in again:
        release(capi, ptr, 100 * mib)
    give_back(capi)
    assert start - free() <= 8 * mib
    large = allocate(capi, 300 * mib)
    release(capi, large, 300 * mib)
    assert start - free() <= 8 * mib
    small = [allocate(capi, 4 * mib) for _ in range(20)]
    for ptr in small:
        release(capi, ptr, 4 * mib)
    assert start - free() <= 72 * mib
    give_back(capi)


def test_many_threads(capi):
    failures = []

    def worker(mark):
        n = 1 << 16
        try:
            for _ in range(60):
                x = allocate(capi, 4 * n)
                capi.check(capi.lib().tcx_hip_fill(0, x, n, float(mark), capi.stream()), "fill")
                host = np.empty(n, np.float32)
                capi.check(capi.lib().tcx_hip_memcpy_d2h(host.ctypes.data, x, 4 * n, capi.stream()), "copy")
                if not (host == mark).all():
                    failures.append(mark)
                release(capi, x, 4 * n)
        except Exception as error:  # noqa: BLE001 - reported by the assertion
            failures.append(error)

    threads = [threading.Thread(target=worker, args=(i + 1,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures
    give_back(capi)
