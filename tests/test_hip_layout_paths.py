"""Gathers, concats and embeddings on the device against NumPy, bit for bit,
where their unit widths and thread shares change."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import require_gpu
from hip_cases import assert_bits

pytestmark = pytest.mark.gpu

DTYPES = ["float32", "int32", "bool"]


@pytest.fixture(scope="module")
def cx():
    require_gpu()
    import tensorcx
    return tensorcx


def values(shape, dtype, seed=1):
    rng = np.random.default_rng(seed)
    if dtype == "bool":
        return rng.random(shape) > 0.5
    words = rng.integers(0, 2**32, shape, dtype=np.uint32)
    return words.view(dtype) if words.ndim else words.reshape(1).view(dtype).reshape(())


def same(actual, expected, what):
    if expected.dtype == np.bool_:
        np.testing.assert_array_equal(actual, expected, what)
    else:
        assert_bits(actual.view(np.int32), np.array(expected, order="C").view(np.int32), what)


# Innermost runs of 16, 4 and single elements; ranks folding to 1-5; 2^18
# units and more (four units a thread) with and without a remainder.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape,axes", [((2, 5, 3, 64), (0, 2, 1, 3)), ((3, 7, 2, 6), (0, 2, 1, 3)), ((4, 9), (1, 0)),
                                        ((2, 3, 4, 5, 16), (4, 2, 0, 1, 3)), ((2, 3, 2, 5, 8), (2, 0, 3, 1, 4)),
                                        ((33, 70, 31, 16), (1, 0, 2, 3)), ((1025, 1027), (1, 0)),
                                        ((16, 67, 16, 64), (0, 2, 1, 3)), ((1, 1, 5), (2, 0, 1)), ((513, 2, 513), (1, 0, 2))])
def test_transpose(cx, dtype, shape, axes):
    x = values(shape, dtype)
    same(cx.transpose(cx.tensor(x, device="hip"), axes).numpy(), np.ascontiguousarray(x.transpose(axes)), f"{shape} {axes}")


@pytest.mark.parametrize("dtype", DTYPES)
def test_slices(cx, dtype):
    x = values((6, 40, 48), dtype)
    h = cx.tensor(x, device="hip")
    for key in [(slice(None), -1), (slice(1, 5), slice(4, 36, 4)), (slice(None), slice(None, None, -1)),
                (slice(None), slice(None), slice(None, None, -1)), (slice(None), slice(None), slice(16, 48)),
                (slice(None), slice(None), slice(1, 33)), (2, 3), (2, 3, 4), (slice(0, 0),), (slice(None), slice(None), 7),
                (slice(None, None, 5), slice(7, 3, -2), slice(4, 44, 3))]:
        same(h[key].numpy(), np.array(x[key], order="C"), f"{key}")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("lead,widths,tail,axis", [((), (3, 4), (5,), 0), ((2,), (64, 1), (16,), 1), ((3, 2), (1023, 1), (64,), 2),
                                                   ((2,), (4, 0, 8), (4,), 1), ((5,), (1, 2, 3, 4, 5, 6, 7, 8, 9, 10), (), 1),
                                                   ((128,), (2047, 1), (16,), 1), ((7,), (300, 200), (513,), 1),
                                                   ((4,), (0, 0), (3,), 1), ((), (100001, 3), (), 0)])
def test_concat(cx, dtype, lead, widths, tail, axis):
    parts = [values(lead + (w,) + tail, dtype, seed) for seed, w in enumerate(widths)]
    got = cx.concat([cx.tensor(p, device="hip") for p in parts], axis)
    same(got.numpy(), np.concatenate(parts, axis), f"{lead} {widths} {tail}")


@pytest.mark.parametrize("width", [0, 1, 3, 4, 8, 64, 100, 128, 1024, 1030, 4100])
@pytest.mark.parametrize("shape", [(1,), (3, 7), (1000,)])
def test_embedding(cx, width, shape):
    rng = np.random.default_rng(width)
    table = values((37, width), "float32")
    ids = rng.integers(0, 37, shape).astype(np.int32)
    h = cx.tensor(table, device="hip")
    same(cx.embedding(cx.tensor(ids, device="hip"), h).numpy(), table[ids], f"{width} {shape}")
    for bad in (-1, 37, 2**31 - 1, -2**31):
        wrong = ids.copy()
        wrong.reshape(-1)[-1] = bad
        with pytest.raises(ValueError):
            cx.embedding(cx.tensor(wrong, device="hip"), h)
    # The check of one call does not carry over to the next.
    same(cx.embedding(cx.tensor(ids, device="hip"), h).numpy(), table[ids], f"{width} {shape} again")


def test_embedding_many_rows(cx):
    table = values((50, 12), "float32")
    ids = np.random.default_rng(3).integers(0, 50, 1_200_000).astype(np.int32)
    h = cx.tensor(table, device="hip")
    same(cx.embedding(cx.tensor(ids, device="hip"), h).numpy(), table[ids], "many rows")
    ids[1_100_001] = 50
    with pytest.raises(ValueError):
        cx.embedding(cx.tensor(ids, device="hip"), h)


@pytest.mark.parametrize("width", [(1 << 28) + 5, (1 << 30) + 8])
def test_embedding_row_wider_than_the_grid(width):
    """A table of one row of more than 2^28 units, words or 16 bytes (the grid
    of whole rows covers 2^28): the last columns are copied too."""
    require_gpu()
    import ctypes

    import tensorcx_hip_capi as capi
    lib, vp, i64 = capi.lib(), ctypes.c_void_p, ctypes.c_int64
    marks = np.arange(1, 17, dtype=np.float32)
    table, out, flag = (capi.DeviceBuffer(4 * n) for n in (width, width, 1))
    capi.check(lib.tcx_hip_fill(0, table.ptr, width, 2.0, capi.stream()), "fill")
    capi.check(lib.tcx_hip_fill(0, out.ptr, width, -7.0, capi.stream()), "fill")
    tail = 4 * (width - marks.size)
    capi.check(lib.tcx_hip_memcpy_h2d(table.address + tail, marks.ctypes.data, marks.nbytes, capi.stream()), "h2d")
    ids = capi.DeviceArray.from_numpy(np.zeros(1, np.int32))
    capi.check(lib.tcx_hip_embedding_f32(vp(ids.ptr), table.ptr, out.ptr, i64(1), i64(1), i64(width), flag.ptr,
                                         vp(capi.stream())), "embedding")
    got = np.empty_like(marks)
    for start, expected in ((tail, marks), (0, np.full(16, 2, np.float32)), (tail // 32 * 16, np.full(16, 2, np.float32))):
        capi.check(lib.tcx_hip_memcpy_d2h(got.ctypes.data, out.address + start, got.nbytes, capi.stream()), "d2h")
        np.testing.assert_array_equal(got, expected)


# Rows by 16 bytes and by words, one and four of them a thread, in blocks that
# they do not fill.
@pytest.mark.parametrize("count,width", [(257, 1), (300_001, 1), (100_003, 3), (70_001, 5), (1023, 255), (1030, 257),
                                         (700_001, 4), (600_001, 12), (2049, 1032), (5000, 1036)])
def test_embedding_packed_rows(cx, count, width):
    rng = np.random.default_rng(count)
    table, ids = values((19, width), "float32"), rng.integers(0, 19, count).astype(np.int32)
    h = cx.tensor(table, device="hip")
    same(cx.embedding(cx.tensor(ids, device="hip"), h).numpy(), table[ids], f"{count} {width}")
    ids[count - 2] = 19
    with pytest.raises(ValueError):
        cx.embedding(cx.tensor(ids, device="hip"), h)
