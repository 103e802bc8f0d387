"""topk on the device against the oracle at the sizes where its selection
changes: rows that are all candidates, the threshold pass, the radix
selection, and the three ways the chosen elements are put in order. Bit-exact
values and indices."""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from conftest import require_gpu
from hip_cases import assert_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cx():
    require_gpu()
    import tensorcx
    return tensorcx


def values_of(kind, shape, rng):
    if kind == "int32":
        return rng.integers(-2**31, 2**31, shape, dtype=np.int64).astype(np.int32)
    if kind == "ties":  # more equal elements than the candidate buffer holds
        return rng.integers(0, 3, shape).astype(np.float32)
    if kind == "equal":
        return np.full(shape, -0.0, np.float32)
    x = rng.standard_normal(shape).astype(np.float32)
    if kind == "special":
        flat = x.reshape(-1)
        at = rng.permutation(flat.size)[: max(8, flat.size // 8)]
        flat[at] = rng.choice(np.array([np.nan, np.inf, -np.inf, 0.0, -0.0], np.float32), at.size)
    return x


def check(cx, x, axis, k, largest, sort):
    values, indices = cx.topk(cx.tensor(x, device="hip"), k, axis, largest, sort)
    expected_values, expected_indices = oracle.topk(x, k, axis, largest, sort)
    what = f"{x.shape} axis={axis} k={k} largest={largest} sorted={sort}"
    assert_bits(indices.numpy(), expected_indices, "indices " + what)
    assert_bits(values.numpy(), expected_values, "values " + what)


# (row length, ks): a wave takes rows up to 1024 and k up to 8 (with 1, 4 or 16
# keys a lane), the direct rows end at 256 or 1024, the threshold pass at k = 64
# or 256, the sort in LDS at k = 1024.
EDGES = [(1, [1]), (63, [1, 8, 63]), (64, [2, 8, 9]), (65, [1, 8, 9]), (256, [1, 8, 64, 256]), (257, [1, 8, 64, 65, 257]),
         (1024, [1, 8, 9, 64, 65, 1024]), (1025, [3, 8, 65, 256, 257, 1025]), (4097, [1, 64, 256, 1024, 1025, 4097]), (8192, [50, 64, 300]),
         (8193, [50, 64, 256, 257]), (20001, [7, 256, 1500])]


@pytest.mark.parametrize("kind", ["normal", "special", "ties", "equal", "int32"])
@pytest.mark.parametrize("n,ks", EDGES, ids=[str(n) for n, _ in EDGES])
def test_row_lengths_and_counts(cx, n, ks, kind):
    rng = np.random.default_rng(n)
    x = values_of(kind, (3, n), rng)
    for k in ks:
        for largest in (True, False):
            for sort in (True, False):
                check(cx, x, -1, k, largest, sort)


@pytest.mark.parametrize("kind", ["normal", "special", "ties", "equal", "int32"])
@pytest.mark.parametrize("shape,axis", [((1, 16384), -1), ((3, 16389), -1), ((2, 65541), -1), ((128, 16385), -1),
                                        ((129, 16385), -1), ((16400, 5), 0)])
def test_rows_in_parts(cx, shape, axis, kind):
    """Few long rows are cut into parts (of lengths that leave a short last
    one); 129 rows and k = 257 are not."""
    x = values_of(kind, shape, np.random.default_rng(shape[0]))
    for k in (1, 50, 256, 257):
        check(cx, x, axis, k, True, True)
    check(cx, x, axis, 50, False, False)


@pytest.mark.parametrize("kind", ["special", "ties"])
def test_other_axes(cx, kind):
    rng = np.random.default_rng(5)
    x = values_of(kind, (2, 1500, 3), rng)
    for k in (1, 40, 70, 300, 1100, 1500):
        check(cx, x, 1, k, True, True)
        check(cx, x, 1, k, False, False)
    short = values_of(kind, (3, 90, 7), rng)
    for k in (1, 8, 9):
        check(cx, short, 1, k, True, True)
        check(cx, short, 1, k, False, False)


def test_unaligned_rows(cx):
    """Rows of an odd length start at every offset from a 16-byte boundary."""
    rng = np.random.default_rng(6)
    for n in (4099, 33001):
        x = values_of("special", (9, n), rng)
        check(cx, x, -1, 50, True, True)


def test_more_rows_than_one_per_compute_unit(cx):
    rng = np.random.default_rng(7)
    check(cx, values_of("special", (3000, 70), rng), -1, 5, True, True)
    check(cx, values_of("ties", (700, 1100), rng), -1, 20, True, False)


# Up to 12 elements: k = 1 (and 2 in 256 threads) in passes, more of them when
# many candidates pass the bound, from rows in one block of 256 or 1024 threads
# and in parts; 13 leave that kernel. 255 rows of 20001 take 1024 threads.
@pytest.mark.parametrize("kind", ["special", "equal", "ordered", "int32"])
@pytest.mark.parametrize("rows,n", [(5, 257), (300, 1025), (255, 20001), (256, 20001), (3, 16389)])
def test_few_elements(cx, rows, n, kind):
    rng = np.random.default_rng(n)
    x = np.sort(values_of("special", (rows, n), rng), axis=-1) if kind == "ordered" else values_of(kind, (rows, n), rng)
    for k in (1, 2, 3, 12, 13):
        check(cx, x, -1, k, True, True)
        check(cx, x, -1, k, False, False)


@pytest.mark.parametrize("k", [1, 3])
def test_ordered_rows_take_little_longer(k):
    """Rows in order pass every bound: they took 14 times as long as rows in no
    order (now at most twice)."""
    require_gpu()
    import ctypes

    import tensorcx_hip_capi as capi
    i64, rows, n = ctypes.c_int64, 4096, 1025
    values, indices = capi.DeviceArray((rows, k)), capi.DeviceArray((rows, k), np.int32)
    start, end, took = capi.Event(), capi.Event(), []
    for x in (np.random.default_rng(1).standard_normal((rows, n), np.float32), np.tile(np.arange(n, dtype=np.float32), (rows, 1))):
        held, best = capi.DeviceArray.from_numpy(x), np.inf
        for _ in range(5):
            start.record()
            for _ in range(10):
                capi.check(capi.lib().tcx_hip_topk(0, *(ctypes.c_void_p(t.ptr) for t in (held, values, indices)), i64(rows),
                                                   i64(n), i64(1), i64(k), 1, 1, ctypes.c_void_p(capi.stream())), "topk")
            end.record()
            end.synchronize()
            best = min(best, start.elapsed_ms(end))
        took.append(best)
    assert took[1] < 5 * took[0], took


# A wave a row up to 2048 elements (k = 3) and, with 2048 or 4096 rows and more,
# up to 16 elements of 1024; more of either, and fewer rows, take a block a row.
@pytest.mark.parametrize("kind", ["special", "equal", "ordered", "int32"])
@pytest.mark.parametrize("rows,n,ks", [(300, 1025, (1, 3, 4)), (256, 2048, (1, 2, 3)), (255, 2048, (3,)), (257, 2049, (3,)),
                                       (2048, 300, (9, 13, 16, 17)), (2050, 1024, (16,)), (2047, 65, (9, 16)), (4096, 65, (9, 16)),
                                       (600, 2500, (13, 16, 17))])
def test_waves_and_blocks(cx, rows, n, ks, kind):
    rng = np.random.default_rng(rows + n)
    x = np.sort(values_of("special", (rows, n), rng), axis=-1) if kind == "ordered" else values_of(kind, (rows, n), rng)
    for k in ks:
        check(cx, x, -1, k, True, True)
        check(cx, x, -1, k, False, False)
