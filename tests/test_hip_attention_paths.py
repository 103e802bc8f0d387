"""The fused attention kernels against the oracle where their dispatch and
their edges lie: few queries (split and unsplit keys), masks of every kind and
broadcast, and special values under them. The bar is the reference test's,
allclose(rtol=2e-4, atol=2e-5)."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle
from conftest import require_gpu
from hip_cases import assert_close

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cx():
    require_gpu()
    import tensorcx
    return tensorcx


def f32(shape, seed):
    return np.random.default_rng(seed).normal(size=shape).astype(np.float32)


def check(cx, q, k, v, mask=None, causal=False):
    args = [cx.tensor(t, device="hip") for t in (q, k, v)]
    held = None if mask is None else cx.tensor(mask, device="hip")
    got = cx.attention(*args, held, is_causal=causal).numpy()
    with np.errstate(all="ignore"):
        expected = oracle.attention(q, k, v, mask, causal)
    assert_close(got, expected, 2e-4, 2e-5, f"{q.shape} x {k.shape} causal={causal}")


def masks(kind, shape, rng):
    """A mask of `shape` that hides about a third of the keys."""
    if kind == "bool":
        return rng.random(shape) > 0.3
    mask = rng.normal(size=shape).astype(np.float32)
    mask[rng.random(shape) < 0.2] = -np.inf
    return mask


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("cols", [1, 63, 64, 65, 127, 128, 255, 256, 257, 1000, 4099])
def test_few_queries(cx, d, rows, cols):
    """One to four queries stream the keys, over one block or (256 keys and
    more for few batch matrices) several; five take the matrix kernel."""
    check(cx, f32((2, 3, rows, d), 1), f32((2, 3, cols, d), 2), f32((2, 3, cols, d), 3))


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("kind", ["bool", "additive"])
def test_few_queries_special_values(cx, d, kind):
    rng = np.random.default_rng(d)
    q, k, v = f32((3, 2, 2, d), 4), f32((3, 2, 700, d), 5), f32((3, 2, 700, d), 6)
    mask = masks(kind, (3, 1, 2, 700), rng)
    mask[1, 0, 0] = False if kind == "bool" else -np.inf   # a row with every key hidden
    mask[2, 0, 1, :400] = False if kind == "bool" else -np.inf  # whole splits hidden
    check(cx, q, k, v, mask)
    q[0, 0, 1, 3] = np.nan
    k[0, 1, 600] = np.inf
    k[2, 0, 5] = -np.inf
    v[1, 1, 650, 7] = np.inf     # shows as inf, or as NaN where its key is hidden
    v[2, 1, 3, 0] = np.nan
    check(cx, q, k, v, mask)
    check(cx, q, k, v)


def test_few_queries_many_batch_matrices(cx):
    q, k, v = f32((1500, 4, 64), 7), f32((1500, 300, 64), 8), f32((1500, 300, 64), 9)
    check(cx, q, k, v)


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("rows,cols", [(64, 64), (65, 63), (130, 129), (200, 320), (256, 191)])
def test_both_tile_lengths(cx, d, causal, rows, cols):
    """32- and 64-key tiles: causal calls of 1024 blocks and more, and few."""
    for batch in (5, 520):
        check(cx, f32((batch, rows, d), 35), f32((batch, cols, d), 36), f32((batch, cols, d), 37), None, causal)


# Padded kernels: multiples of eight features, the first and last of each
# kernel's range among them; 8, 66 and 136 keep the unfused route.
@pytest.mark.parametrize("d", [16, 24, 40, 56, 72, 80, 120, 8, 66, 136])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("batch,rows,cols", [(3, 1, 700), (3, 4, 33), (2, 37, 1500), (5, 130, 129), (300, 64, 64)])
def test_padded_features(cx, d, causal, batch, rows, cols):
    q, k, v = f32((batch, rows, d), 41), f32((batch, cols, d), 42), f32((batch, cols, d), 43)
    check(cx, q, k, v, None, causal)
    rng = np.random.default_rng(d)
    for kind in ("bool", "additive"):
        mask = masks(kind, (batch, 1, cols), rng)
        mask[..., cols // 2:] = False if kind == "bool" else -np.inf
        check(cx, q, k, v, mask, causal)


@pytest.mark.parametrize("d", [16, 48, 80])
@pytest.mark.parametrize("rows", [2, 70])
def test_padded_features_special_values(cx, d, rows):
    """Infinities in the first chunk (which padding lanes read) and the last."""
    q, k, v = f32((4, rows, d), 44), f32((4, 900, d), 45), f32((4, 900, d), 46)
    k[0, 5, 0] = np.inf
    k[1, 800, d - 1] = -np.inf
    v[2, 850, 0] = np.inf
    v[3, 3, d - 1] = np.nan
    q[3, 1, 0] = np.inf
    for causal in (False, True):
        check(cx, q, k, v, None, causal)
    mask = np.ones((4, 1, 900), dtype=bool)
    mask[:, :, 600:] = False
    check(cx, q, k, v, mask)


# (batch matrices, rows, cols): one wave for up to 16 queries; four or eight
# waves, whole or split, with splits that end in the middle of a key tile and
# causal parts that are empty.
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("batch,rows,cols", [(3, 5, 4097), (4, 16, 1000), (4, 17, 1000), (2, 64, 2050), (3, 130, 1500),
                                             (4, 512, 515), (70, 16, 200), (20, 129, 700), (256, 16, 33)])
def test_split_keys(cx, d, causal, batch, rows, cols):
    q, k, v = f32((batch, rows, d), 26), f32((batch, cols, d), 27), f32((batch, cols, d), 28)
    check(cx, q, k, v, None, causal)


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_split_keys_special_values(cx, d, causal):
    q, k, v = f32((2, 90, d), 29), f32((2, 1300, d), 30), f32((2, 1300, d), 31)
    q[0, 3, 7] = np.nan
    k[0, 1200] = np.inf
    k[0, 60] = -np.inf
    v[1, 1250, 5] = np.nan   # in the last split, behind the causal mask of every query
    v[1, 40, 6] = np.inf
    check(cx, q, k, v, None, causal)
    mask = masks("additive", (2, 90, 1300), np.random.default_rng(6))
    mask[1, 5] = -np.inf
    mask[0, 9, 100:] = -np.inf
    check(cx, q, k, v, mask, causal)


# Mask shapes against scores of (2, 3, rows, cols): shared, for each batch,
# for each head, for each key, for each query, full.
SHAPES = [lambda r, c: (r, c), lambda r, c: (2, 1, 1, c), lambda r, c: (1, 3, r, c), lambda r, c: (c,),
          lambda r, c: (2, 3, r, 1), lambda r, c: (2, 3, r, c)]


@pytest.mark.parametrize("kind", ["bool", "additive"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d,rows,cols", [(32, 70, 31), (64, 64, 64), (64, 65, 33), (128, 130, 257), (128, 1, 300),
                                         (64, 4, 129), (32, 17, 1)])
def test_masks(cx, d, rows, cols, causal, kind):
    rng = np.random.default_rng(rows * cols)
    q, k, v = f32((2, 3, rows, d), 11), f32((2, 3, cols, d), 12), f32((2, 3, cols, d), 13)
    for shape in SHAPES:
        check(cx, q, k, v, masks(kind, shape(rows, cols), rng), causal)


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("kind", ["bool", "additive"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("rows", [40, 130])
def test_hidden_ends(cx, d, kind, causal, rows):
    """Key masks that hide whole tiles in front and behind, all keys, or all but
    one; values there that are not finite show as NaN all the same. The few
    queries of 16 matrices also split the keys."""
    cols = 700
    q, k, v = f32((8, 2, rows, d), 32), f32((8, 2, cols, d), 33), f32((8, 2, cols, d), 34)
    shown = np.zeros((8, 1, 1, cols), bool)
    for b, (first, end) in enumerate([(0, 700), (0, 31), (0, 64), (0, 65), (300, 500), (699, 700), (0, 0), (95, 97)]):
        shown[b, 0, 0, first:end] = True
    shown[4, 0, 0, 350:400] = False
    mask = shown if kind == "bool" else np.where(shown, np.float32(0.5), np.float32(-np.inf))
    check(cx, q, k, v, mask, causal)
    v[1, 0, 699, 3] = np.nan
    v[1, 1, 33, 4] = np.inf
    v[4, 0, 0, 5] = -np.inf
    v[4, 1, 550, 6] = np.nan
    v[5, 0, 10, 7] = np.inf
    v[6, 1, 640, 8] = np.nan
    check(cx, q, k, v, mask, causal)


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("kind", ["bool", "additive"])
def test_mask_special_values(cx, d, kind):
    rng = np.random.default_rng(3)
    q, k, v = f32((2, 90, d), 14), f32((2, 110, d), 15), f32((2, 110, d), 16)
    mask = masks(kind, (2, 90, 110), rng)
    mask[0, 5] = False if kind == "bool" else -np.inf
    if kind == "additive":
        mask[1, 7, 3], mask[1, 8, 4] = np.nan, np.inf
    q[0, 3, 7] = np.nan
    k[0, 11] = np.inf
    k[0, 12] = -np.inf
    v[1, 80, 5] = np.nan
    v[1, 109, 6] = np.inf
    for causal in (False, True):
        check(cx, q, k, v, mask, causal)


def test_mask_over_nine_batch_axes(cx):
    """Alternating broadcast axes fold to at most eight; nine take the
    unfused route, whose own limit refuses them."""
    lead = (2, 1, 2, 1, 2, 1, 2, 2)
    q, k, v = f32(lead + (3, 32), 17), f32(lead + (5, 32), 18), f32(lead + (5, 32), 19)
    rng = np.random.default_rng(4)
    check(cx, q, k, v, masks("bool", (2, 1, 1, 1, 2, 1, 1, 2, 3, 5), rng))


class Desc(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int64) for n in ("batch", "rows", "cols", "features")] + [
        ("scale", ctypes.c_float), ("causal", ctypes.c_int32), ("mask_kind", ctypes.c_int32),
        ("mask_rank", ctypes.c_int32), ("mask_shape", ctypes.c_int64 * 8), ("mask_strides", ctypes.c_int64 * 8),
        ("mask_row_stride", ctypes.c_int64), ("mask_col_stride", ctypes.c_int64)]


def fused(capi, q, k, v, mask, desc):
    """The C entry on device copies, without a workspace; the mask starts one
    element past a 16-byte boundary."""
    held = [capi.DeviceArray.from_numpy(t) for t in (q, k, v)]
    store = capi.DeviceArray.from_numpy(np.concatenate([np.zeros(1, mask.dtype), mask.reshape(-1)]))
    out = capi.DeviceArray(q.shape)
    capi.check(capi.lib().tcx_hip_flash_attention_f32_ws(
        *(ctypes.c_void_p(t.ptr) for t in held), ctypes.c_void_p(out.ptr),
        ctypes.c_void_p(store.ptr + mask.itemsize), ctypes.byref(desc), None, ctypes.c_size_t(0),
        ctypes.c_void_p(capi.stream())), "attention")
    capi.synchronize()
    return out.numpy()


@pytest.mark.parametrize("kind", ["bool", "additive"])
@pytest.mark.parametrize("rows", [2, 40])
def test_mask_at_an_odd_address(cx, rows, kind):
    import tensorcx_hip_capi as capi
    q, k, v = f32((2, rows, 64), 20), f32((2, 300, 64), 21), f32((2, 300, 64), 22)
    mask = masks(kind, (2, rows, 300), np.random.default_rng(5))
    desc = Desc(batch=2, rows=rows, cols=300, features=64, scale=0.125, mask_kind=1 if kind == "bool" else 2,
                mask_rank=1, mask_row_stride=300, mask_col_stride=1)
    desc.mask_shape[0], desc.mask_strides[0] = 2, rows * 300
    assert_close(fused(capi, q, k, v, mask, desc), oracle.attention(q, k, v, mask), 2e-4, 2e-5, "odd address")
    desc.mask_shape[0] = 3
    with pytest.raises(capi.HipError):
        fused(capi, q, k, v, mask, desc)


@pytest.mark.parametrize("rows", [1, 3])
def test_without_a_workspace(cx, rows):
    """The C entry without a workspace, or with one too small, keeps the keys
    of a matrix in one block."""
    import tensorcx_hip_capi as capi
    lib = capi.lib()
    q, k, v = f32((2, rows, 64), 23), f32((2, 900, 64), 24), f32((2, 900, 64), 25)
    dq, dk, dv = (capi.DeviceArray.from_numpy(t) for t in (q, k, v))
    out = capi.DeviceArray(q.shape)
    capi.flash_attention(dq.ptr, dk.ptr, dv.ptr, out.ptr, 2, rows, 900, 64, 0.125, False)
    capi.synchronize()
    assert_close(out.numpy(), oracle.attention(q, k, v), 2e-4, 2e-5, "no workspace")
    assert lib.tcx_hip_flash_attention_f32_ws(None, None, None, None, None, None, None, ctypes.c_size_t(0),
                                              None) == capi.TCX_INVALID_ARGUMENT


# With q = 0 the additive mask holds the scores, exactly: one key at 0, one at
# -x, the others hidden. The output is then exp(-x) / (1 + exp(-x)): two to four
# ulp of expf, the sum and the division. Both keys in one tile, and so far apart
# that the states of lane groups, tiles or splits have to be joined.
@pytest.mark.parametrize("d", [16, 64, 128])
@pytest.mark.parametrize("rows", [1, 4, 5, 40])
@pytest.mark.parametrize("cols", [2, 90, 700, 4100])
def test_exponentials(cx, d, rows, cols):
    x = np.linspace(0.3, 87, 48).astype(np.float32)
    q, k, v = np.zeros((48, rows, d), np.float32), f32((48, cols, d), 47), np.zeros((48, cols, d), np.float32)
    for first, last in ((0, cols - 1), (cols - 1, 0)):
        mask = np.full((48, 1, cols), -np.inf, np.float32)
        mask[:, 0, first], mask[:, 0, last] = 0, -x
        v[:] = 0
        v[:, last, 1:] = 1
        got = cx.attention(*(cx.tensor(t, device="hip") for t in (q, k, v)), cx.tensor(mask, device="hip")).numpy()
        p = np.exp(-x.astype(np.float64))
        expected = np.broadcast_to((p / (1 + p))[:, None, None], (48, rows, d - 1))
        assert np.abs(got[:, :, 1:] / expected - 1).max() <= 8 * 2.0**-24, (first, last)
        assert not got[:, :, 0].any()
        # Below the normal numbers a probability is still no zero to an
        # infinite value, down to the last one that expf gives.
        mask[:, 0, last] = -np.linspace(87.4, 103, 48).astype(np.float32)
        v[:, last, 3] = np.inf
        got = cx.attention(*(cx.tensor(t, device="hip") for t in (q, k, v)), cx.tensor(mask, device="hip")).numpy()
        assert (got[:, :, 3] == np.inf).all() and np.isfinite(got[:, :, :3]).all()


class SoftmaxDesc(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int64 * 8) for n in ("shape", "score_strides", "mask_strides")] + [
        ("rank", ctypes.c_int32), ("mask_kind", ctypes.c_int32), ("causal", ctypes.c_int32), ("scale", ctypes.c_float)]


def unfused(capi, q, k, v, mask, scale):
    """The two products and the softmax between them."""
    batch, rows, d = q.shape
    cols = k.shape[1]
    dq, dk, dv, dm = (capi.DeviceArray.from_numpy(t) for t in (q, k, v, mask))
    scores, out = capi.DeviceArray((batch, rows, cols)), capi.DeviceArray(q.shape)
    capi.gemm(dq.ptr, dk.ptr, scores.ptr, capi.gemm_desc(rows, cols, d, batch_shape=(batch,), lhs_batch_strides=(rows * d,),
                                                         rhs_batch_strides=(cols * d,), rhs_transposed=True))
    desc = SoftmaxDesc(rank=3, mask_kind=2, scale=scale)
    for i, (n, stride) in enumerate(zip(scores.shape, (rows * cols, cols, 1))):
        desc.shape[i], desc.score_strides[i], desc.mask_strides[i] = n, stride, stride
    capi.check(capi.lib().tcx_hip_attention_softmax_f32(*(ctypes.c_void_p(t.ptr) for t in (scores, dm, scores)),
                                                        ctypes.byref(desc), ctypes.c_void_p(capi.stream())), "softmax")
    capi.gemm(scores.ptr, dv.ptr, out.ptr, capi.gemm_desc(rows, d, cols, batch_shape=(batch,), lhs_batch_strides=(rows * cols,),
                                                          rhs_batch_strides=(cols * d,)))
    capi.synchronize()
    return out.numpy()


@pytest.mark.parametrize("d", [16, 32, 48, 64, 80, 128])
def test_masked_error_against_64_bits(cx, d):
    """The masked and padded kernels are no less exact than the products and
    the softmax that they replace: relative errors (2-norm) over at least 25000
    outputs of each shape, whose ratio one sample moves by 2 % or so."""
    import tensorcx_hip_capi as capi
    ratios = []
    for batch, rows, cols in ((1500, 1, 100), (1500, 1, 700), (500, 3, 300), (100, 16, 200), (50, 40, 128), (20, 130, 600)):
        rng = np.random.default_rng(rows + cols + d)
        q, k, v = f32((batch, rows, d), 51), f32((batch, cols, d), 52), f32((batch, cols, d), 53)
        mask = rng.standard_normal((batch, rows, cols)).astype(np.float32)
        mask[rng.random(mask.shape) < 0.2] = -np.inf
        scale = np.float32(1 / np.sqrt(d))
        s = q.astype(np.float64) @ np.swapaxes(k, 1, 2) * scale + mask
        p = np.exp(s - s.max(-1, keepdims=True))
        exact = p / p.sum(-1, keepdims=True) @ v.astype(np.float64)
        got = cx.attention(*(cx.tensor(t, device="hip") for t in (q, k, v)), cx.tensor(mask, device="hip")).numpy()
        ratios.append(np.linalg.norm(got - exact) / np.linalg.norm(unfused(capi, q, k, v, mask, scale) - exact))
    assert max(ratios) <= 1.03 and np.mean(ratios) <= 0.9, ratios


@pytest.mark.parametrize("rows", [1, 5])
def test_more_matrices_than_a_launch_holds(rows):
    """2^24 + 5 matrices of one key (HIP counts 2^32 work-items a launch), on the
    streaming and on the matrix kernel; the last ones under the last entries of
    a mask with an axis of its own for each half of them."""
    require_gpu()
    import tensorcx_hip_capi as capi
    lib, vp, n, tail, d = capi.lib(), ctypes.c_void_p, (1 << 24) + 6, 64, 16
    q, out = capi.DeviceBuffer(4 * n * rows * d), capi.DeviceBuffer(4 * n * rows * d)
    k, v, mask = capi.DeviceBuffer(4 * n * d), capi.DeviceBuffer(4 * n * d), capi.DeviceBuffer(n)
    for t, size, value in ((q, n * rows * d, 1.0), (k, n * d, 1.0), (v, n * d, 2.0), (out, n * rows * d, -7.0)):
        capi.check(lib.tcx_hip_fill(0, t.ptr, size, value, capi.stream()), "fill")
    capi.check(lib.tcx_hip_fill(2, mask.ptr, n, 1.0, capi.stream()), "fill")
    marks, shown = f32((tail, d), 61), np.arange(tail) % 3 != 0
    for t, host, at in ((v, marks, 4 * (n - tail) * d), (mask, shown.astype(np.uint8), n - tail)):
        capi.check(lib.tcx_hip_memcpy_h2d(t.address + at, host.ctypes.data, host.nbytes, capi.stream()), "h2d")
    desc = Desc(batch=n, rows=rows, cols=1, features=d, scale=0.25, mask_kind=1, mask_rank=2, mask_row_stride=0, mask_col_stride=1)
    desc.mask_shape[0], desc.mask_shape[1], desc.mask_strides[0], desc.mask_strides[1] = 2, n // 2, n // 2, 1
    capi.check(lib.tcx_hip_flash_attention_f32_ws(q.ptr, k.ptr, v.ptr, out.ptr, mask.ptr, ctypes.byref(desc), None,
                                                  ctypes.c_size_t(0), vp(capi.stream())), "attention")
    got = np.empty((tail, rows, d), np.float32)
    expected = np.repeat(np.where(shown[:, None], marks, np.float32(0))[:, None], rows, 1)
    for first, want in ((n - tail, expected), (0, np.full_like(got, 2)), ((1 << 24) - tail, np.full_like(got, 2))):
        capi.check(lib.tcx_hip_memcpy_d2h(got.ctypes.data, out.address + 4 * first * rows * d, got.nbytes, capi.stream()), "d2h")
        want = want.copy()
        if first != n - tail and first + tail > n - tail:
            want[n - tail - first:] = expected[:first + tail - (n - tail)]
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("batch,rows,cols,d", [(4, 256, 256, 64), (2, 64, 1500, 128), (8, 1, 2100, 32), (3, 17, 1000, 80)])
@pytest.mark.parametrize("causal", [False, True])
def test_workspace_with_room_for_some_splits(cx, batch, rows, cols, d, causal):
    """The keys are split as far as the workspace goes, and what lies behind it
    stays as it is."""
    import tensorcx_hip_capi as capi
    q, k, v = f32((batch, rows, d), 62), f32((batch, cols, d), 63), f32((batch, cols, d), 64)
    held = [capi.DeviceArray.from_numpy(t) for t in (q, k, v)]
    desc = Desc(batch=batch, rows=rows, cols=cols, features=d, scale=d ** -0.5, causal=int(causal))
    query = capi.lib().tcx_hip_flash_attention_workspace_bytes
    query.restype = ctypes.c_size_t
    full, expected = query(ctypes.byref(desc)), oracle.attention(q, k, v, None, causal)
    for nbytes in {full, full // 2, full // 3, 1000, 0}:
        out = capi.DeviceArray(q.shape)
        workspace = capi.DeviceArray.from_numpy(np.full(nbytes // 4 + 64, 99, np.float32))
        capi.check(capi.lib().tcx_hip_flash_attention_f32_ws(
            *(ctypes.c_void_p(t.ptr) for t in (*held, out)), None, ctypes.byref(desc), ctypes.c_void_p(workspace.ptr),
            ctypes.c_size_t(nbytes), ctypes.c_void_p(capi.stream())), "attention")
        capi.synchronize()
        assert_close(out.numpy(), expected, 2e-4, 2e-5, f"{nbytes} of {full} bytes")
        assert (workspace.numpy()[nbytes // 4:] == 99).all()


# Eight waves and 64-key tiles (tests of the plan pin that these sizes take
# them): query and key remainders, and values that are not finite in the last,
# partial key tile and in rows of every wave.
@pytest.mark.parametrize("batch,rows,cols", [(64, 300, 300), (32, 1000, 1000), (40, 500, 500), (32, 970, 1025)])
def test_eight_waves(cx, batch, rows, cols):
    q, k, v = f32((batch, rows, 128), 65), f32((batch, cols, 128), 66), f32((batch, cols, 128), 67)
    check(cx, q, k, v)
    q[0, ::37, 5] = np.nan
    k[1, cols - 1, 3] = np.inf
    k[2, 70, 4] = -np.inf
    v[3, cols - 1, 127] = np.inf
    v[3, 64, 2] = np.nan
    v[batch - 1, 0, 0] = -np.inf
    q[1, rows - 1] = 0
    check(cx, q, k, v)
