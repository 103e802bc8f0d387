"""Exported storage after its release: kept by its pool for an allocation of
the same size that waits for all work on the device, within the pool's limits,
given back with the pool's blocks, and taken by one owner at a time. Without a
pool, and in one that may keep nothing, it is freed."""

from __future__ import annotations

import contextlib
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
    return ptr, owner


def release(capi, block, nbytes):
    capi.lib().tcx_hip_release_uncached(block[0], nbytes, block[1])


@contextlib.contextmanager
def pool_of(capi, nbytes, blocks):
    pool = ctypes.c_void_p()
    capi.check(capi.lib().tcx_hip_pool_create(nbytes, blocks, None, ctypes.byref(pool)), "pool")
    capi.check(capi.lib().tcx_hip_pool_enter(pool), "enter")
    try:
        yield pool
    finally:
        capi.check(capi.lib().tcx_hip_pool_exit(pool), "exit")
        capi.lib().tcx_hip_pool_destroy(pool)


def stats(capi, pool):
    out = capi.PoolStats()
    capi.check(capi.lib().tcx_hip_pool_stats(pool, ctypes.byref(out)), "stats")
    return out


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
    with pool_of(capi, 8 * n, 4):
        for attempt in range(3):
            x = allocate(capi, 4 * n)
            capi.check(capi.lib().tcx_hip_fill(0, x[0], n, float(attempt + 1), capi.stream()), "fill")
            capi.synchronize()
            for _ in range(30):  # some milliseconds in front of the read
                capi.gemm(a.ptr, b.ptr, c.ptr, capi.gemm_desc(2048, 2048, 2048), stream)
            capi.check(capi.lib().tcx_hip_scalar_op(1, 0, x[0], copy.ptr, n, 0.0, 0, stream), "copy")
            release(capi, x, 4 * n)
            y = allocate(capi, 4 * n)
            assert y[0].value == x[0].value  # kept, and the newest of its size
            capi.check(capi.lib().tcx_hip_fill(0, y[0], n, -1.0, capi.stream()), "fill")
            capi.synchronize()
            capi.check(capi.lib().tcx_hip_stream_synchronize(stream), "synchronize")
            np.testing.assert_array_equal(copy.numpy(), np.full(n, attempt + 1, np.float32))
            release(capi, y, 4 * n)


MIB = 1 << 20


def free_bytes(capi):
    return capi.device_info()["free_bytes"]


def test_bounds_and_giving_back(capi):
    start = free_bytes(capi)
    with pool_of(capi, 512 * MIB, 16) as pool:
        blocks = [allocate(capi, 100 * MIB) for _ in range(8)]
        for block in blocks:
            release(capi, block, 100 * MIB)
        assert 0 < start - free_bytes(capi) <= 520 * MIB  # five of the eight are kept
        s = stats(capi, pool)
        assert (s.cached_blocks, s.uncached_returns, s.free_calls) == (0, 8, 3)
        again = [allocate(capi, 100 * MIB) for _ in range(8)]
        assert {p.value for p, _ in again[:5]} == {p.value for p, _ in blocks[3:]}
        for block in again:
            release(capi, block, 100 * MIB)
        capi.check(capi.lib().tcx_hip_pool_trim(pool), "trim")
        assert start - free_bytes(capi) <= 8 * MIB
        large = allocate(capi, 600 * MIB)
        release(capi, large, 600 * MIB)
        assert start - free_bytes(capi) <= 8 * MIB
        small = [allocate(capi, 4 * MIB) for _ in range(20)]
        for block in small:
            release(capi, block, 4 * MIB)
        assert 0 < start - free_bytes(capi) <= 72 * MIB  # sixteen
    assert start - free_bytes(capi) <= 8 * MIB


def test_cached_blocks_come_first(capi):
    """Exported blocks make room for cached ones, the oldest first."""
    start = free_bytes(capi)
    with pool_of(capi, 300 * MIB, 8) as pool:
        blocks = [allocate(capi, n * MIB) for n in (100, 101, 102)]
        for block, n in zip(blocks[:2], (100, 101)):
            release(capi, block, n * MIB)
        capi.lib().tcx_hip_release(blocks[2][0], 102 * MIB, blocks[2][1])  # 303 MiB: the first goes
        s = stats(capi, pool)
        assert (s.cached_blocks, s.cached_bytes, s.free_calls) == (1, 102 * MIB, 1)
        assert start - free_bytes(capi) <= 211 * MIB
        again = allocate(capi, 101 * MIB)
        assert again[0].value == blocks[1][0].value
        release(capi, again, 101 * MIB)


@pytest.mark.parametrize("pooled", [False, True])
def test_nothing_kept_outside_the_limits(capi, pooled):
    """Without a pool, and with one whose limit is 0 bytes."""
    start = free_bytes(capi)
    with pool_of(capi, 0, 16) if pooled else contextlib.nullcontext():
        blocks = [allocate(capi, 64 * MIB) for _ in range(4)]
        assert start - free_bytes(capi) >= 250 * MIB
        for block in blocks:
            release(capi, block, 64 * MIB)
        assert start - free_bytes(capi) <= 8 * MIB


def test_release_after_the_pool_was_left(capi):
    start = free_bytes(capi)
    with pool_of(capi, 256 * MIB, 16):
        block = allocate(capi, 64 * MIB)
    release(capi, block, 64 * MIB)
    assert start - free_bytes(capi) <= 8 * MIB


def test_many_threads(capi):
    """A pool for each thread, whose blocks other threads release."""
    failures = []
    n, ready = 1 << 16, threading.Barrier(8)
    handed = [[] for _ in range(8)]

    def worker(mark):
        try:
            with pool_of(capi, 16 * n, 4):
                for turn in range(60):
                    x = allocate(capi, 4 * n)
                    capi.check(capi.lib().tcx_hip_fill(0, x[0], n, float(mark), capi.stream()), "fill")
                    host = np.empty(n, np.float32)
                    capi.check(capi.lib().tcx_hip_memcpy_d2h(host.ctypes.data, x[0], 4 * n, capi.stream()), "copy")
                    if not (host == mark).all():
                        failures.append(mark)
                    if turn % 3:
                        release(capi, x, 4 * n)
                    else:
                        handed[mark - 1].append(x)
                        other = handed[mark % 8]
                        while other:
                            release(capi, other.pop(), 4 * n)
                ready.wait(60)
        except Exception as error:  # noqa: BLE001 - reported by the assertion
            failures.append(error)

    threads = [threading.Thread(target=worker, args=(i + 1,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for blocks in handed:
        for block in blocks:
            release(capi, block, 4 * n)
    assert not failures
