"""Matrix products whose rows are not 16-byte: K or N no multiple of four, or
operands off a 16-byte boundary, on every kernel that takes them. The bar is
the matmul bar against float64; infinities in neighbouring rows and columns
must not leak into an output that does not use them."""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from conftest import require_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    require_gpu()
    import tensorcx_hip_capi
    return tensorcx_hip_capi


def shifted(capi, array, shift):
    """A device copy that starts `shift` floats past an aligned address."""
    store = capi.DeviceArray.from_numpy(np.concatenate([np.full(shift, np.nan, np.float32), array.reshape(-1)]))
    return store, store.ptr + 4 * shift


def product(capi, a, b, trans, bias=None, shift=0, workspace=False):
    batch = a.shape[:-2]
    m, k = a.shape[-2:]
    n = b.shape[-2] if trans else b.shape[-1]
    held_a, pa = shifted(capi, a, shift)
    held_b, pb = shifted(capi, b, shift)
    out = capi.DeviceArray((shift + int(np.prod(batch, dtype=np.int64)) * m * n + 8,))
    capi.check(capi.lib().tcx_hip_fill(0, out.ptr, out.size, -7.0, capi.stream()), "fill")
    held_bias = capi.DeviceArray.from_numpy(bias) if bias is not None else None
    desc = capi.gemm_desc(m, n, k, batch_shape=batch, lhs_batch_strides=(m * k,) * len(batch),
                          rhs_batch_strides=(k * n,) * len(batch), rhs_transposed=trans,
                          bias=held_bias.ptr if held_bias is not None else None)
    ws = capi.gemm_workspace(desc) if workspace else None
    capi.gemm(pa, pb, out.ptr + 4 * shift, desc, workspace=ws)
    capi.synchronize()
    got = out.numpy()
    assert (got[:shift] == -7.0).all() and (got[-8:] == -7.0).all()  # nothing outside the output
    return got[shift:-8].reshape(batch + (m, n))


def reference(a, b, trans, bias):
    with np.errstate(all="ignore"):
        y = a.astype(np.float64) @ (np.swapaxes(b, -1, -2) if trans else b).astype(np.float64)
    return y if bias is None else y + bias


def check(capi, m, n, k, trans, *, batch=(), shift=0, workspace=False, leak=True):
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    a = rng.standard_normal(batch + (m, k)).astype(np.float32)
    b = rng.standard_normal(batch + ((n, k) if trans else (k, n))).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    what = f"{batch} {m}x{n}x{k} trans={trans} shift={shift}"
    got = product(capi, a, b, trans, bias, shift, workspace)
    error = np.abs(got - reference(a, b, trans, bias)).max()
    assert error <= 1e-4 * np.sqrt(k), f"{what}: {error}"
    if not leak or m < 3 or n < 3:
        return
    # A row of A and a row of W (a column of B) of infinities and NaN.
    a[..., 1, :] = np.inf
    if trans:
        b[..., 1, :] = np.nan
    else:
        b[..., :, 0] = np.inf
        b[..., :, n - 1] = np.nan
    got = product(capi, a, b, trans, bias, shift, workspace)
    clean = np.ones((m, n), bool)
    clean[1] = False
    if trans:
        clean[:, 1] = False
    else:
        clean[:, 0] = clean[:, n - 1] = False
    expected = reference(a, b, trans, bias)
    error = np.abs(got[..., clean] - expected[..., clean]).max()
    assert error <= 1e-4 * np.sqrt(k), f"{what} next to infinities: {error}"
    assert not np.isfinite(got[..., ~clean]).any(), what


@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("k", [5, 6, 7, 63, 65, 66, 67, 127, 129, 191, 194, 255, 321])
def test_direct_tiles(capi, trans, k):
    """64x64 tiles (9 x 15 of them): k tiles of 64 cut at every remainder, from
    one to six of them; and the 32x64 tiles of a short last round."""
    check(capi, 130, 261, k, trans, batch=(9,))
    check(capi, 130, 261, k, trans, batch=(19,), leak=False)


@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("n", [705, 706, 707, 708, 641])
@pytest.mark.parametrize("k", [128, 130])
def test_direct_columns(capi, trans, n, k):
    check(capi, 700, n, k, trans)


@pytest.mark.parametrize("trans", [False, True])
def test_direct_many_tiles(capi, trans):
    check(capi, 2050, 2049, 70, trans)
    check(capi, 2050, 2048, 71, trans, leak=False)
    check(capi, 1030, 1027, 4099, trans, workspace=True, leak=False)  # 81 tiles of 128x128: the workspace is left alone


@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("m,n", [(64, 64), (33, 65), (97, 31), (142, 321), (200, 2), (5, 7), (40, 33), (64, 129)])
@pytest.mark.parametrize("k", [5, 17, 30, 225, 739, 1030])
def test_small_tiles(capi, trans, m, n, k):
    check(capi, m, n, k, trans)


@pytest.mark.parametrize("m", [2, 3, 16, 17, 32])
@pytest.mark.parametrize("k", [6, 61, 65, 707, 2049, 4098])
def test_skinny(capi, m, k):
    """At most 32 rows of A against W, and at most 32 columns of B."""
    for n in (256, 438, 5001):
        check(capi, m, n, k, True)
    check(capi, 300, m, k, False)
    check(capi, 300, m, k, True)


@pytest.mark.parametrize("k", [64, 65, 255, 1025, 3245, 9999])
def test_vectors(capi, k):
    for n in (1, 3, 264, 1001):
        check(capi, 1, n, k, True, leak=False)
    check(capi, 517, 1, k, False, leak=False)
    check(capi, 1, 37, k, True, batch=(5,), leak=False)


@pytest.mark.parametrize("shift", [1, 2, 3])
@pytest.mark.parametrize("trans", [False, True])
def test_unaligned_operands(capi, trans, shift):
    """Sizes of 16-byte rows at addresses between them."""
    for m, n, k in ((700, 704, 128), (64, 64, 256), (16, 512, 1024), (1, 300, 512), (1100, 1100, 260)):
        check(capi, m, n, k, trans, shift=shift, leak=False)


# Zero-padded copies in the workspace: 16 x 16 tiles of 128 x 128 (one full
# round), and less than 128 k whatever the last round; without them 17 x 16 and
# 24 x 24 tiles, whose last round is a small part of one.
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("m,n,k,padded", [(2048, 2047, 1027, True), (5760, 5888, 127, True), (2048, 2049, 1026, False),
                                          (3000, 3001, 1000, False)])
def test_padded_copies(capi, m, n, k, padded, trans):
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((n, k) if trans else (k, n)).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    da, db, dbias, out = (capi.DeviceArray.from_numpy(t) for t in (a, b, bias, np.empty((m, n), np.float32)))
    linear = None
    for act in ("none", "silu", "gelu"):
        desc = capi.gemm_desc(m, n, k, rhs_transposed=trans, bias=dbias.ptr, activation=act)
        workspace = capi.gemm_workspace(desc)
        words = workspace.nbytes // 4
        capi.check(capi.lib().tcx_hip_fill(0, workspace.ptr, words, 99.0, capi.stream()), "fill")
        capi.gemm(da.ptr, db.ptr, out.ptr, desc, workspace=workspace)
        used = np.empty(words, np.float32)
        capi.check(capi.lib().tcx_hip_memcpy_d2h(used.ctypes.data, workspace.ptr, 4 * words, capi.stream()), "copy")
        assert (used != 99).any() == padded
        got = out.numpy()
        if linear is None:
            linear = got
            error = np.abs(got - reference(a, b, trans, bias)).max()
            assert error <= 1e-4 * np.sqrt(k), error
        else:  # the same product, so the activation meets the same bits
            np.testing.assert_allclose(got, getattr(oracle, act)(linear), rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("m,n,k", [(2708, 4, 440), (5000, 7, 260), (8000, 32, 129), (20000, 17, 1001), (30000, 2, 64)])
def test_tall_and_narrow(capi, m, n, k):
    """At most 32 columns of a [k, n] B, with one to eight waves a block."""
    check(capi, m, n, k, False, shift=1, leak=False)


@pytest.mark.parametrize("trans", [False, True])
def test_more_rows_than_a_launch_holds(capi, trans):
    """2^26 + 70 rows of 65 k by one column: a wave each would be more
    work-items than HIP counts."""
    rows, k, tail = (1 << 26) + 70, 65, 200
    rng = np.random.default_rng(5)
    a, b, out = capi.DeviceBuffer(4 * rows * k), capi.DeviceArray.from_numpy(rng.standard_normal(k).astype(np.float32)), \
        capi.DeviceBuffer(4 * rows)
    capi.check(capi.lib().tcx_hip_fill(0, a.ptr, rows * k, 1.0, capi.stream()), "fill")
    capi.check(capi.lib().tcx_hip_fill(0, out.ptr, rows, -7.0, capi.stream()), "fill")
    last = rng.standard_normal((tail, k)).astype(np.float32)
    capi.check(capi.lib().tcx_hip_memcpy_h2d(a.address + 4 * (rows - tail) * k, last.ctypes.data, last.nbytes, capi.stream()), "h2d")
    m, n = (1, rows) if trans else (rows, 1)
    lhs, rhs = (b.ptr, a.ptr) if trans else (a.ptr, b.ptr)
    capi.gemm(lhs, rhs, out.ptr, capi.gemm_desc(m, n, k, rhs_transposed=trans))
    got = np.empty(tail, np.float32)
    column = b.numpy().astype(np.float64)
    for first, expected in ((rows - tail, last @ column), (0, np.full(tail, column.sum())),
                            ((1 << 25) + 7, np.full(tail, column.sum()))):
        capi.check(capi.lib().tcx_hip_memcpy_d2h(got.ctypes.data, out.address + 4 * first, got.nbytes, capi.stream()), "d2h")
        assert np.abs(got - expected).max() <= 1e-4 * np.sqrt(k)
