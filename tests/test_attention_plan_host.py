"""How fused attention would run a call (tcx_hip_flash_attention_plan): the
kernel, its form and its split of the keys. No kernel runs here."""

from __future__ import annotations

import ctypes

import pytest

import tensorcx_hip_capi as capi


class Desc(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int64) for n in ("batch", "rows", "cols", "features")] + [
        ("scale", ctypes.c_float), ("causal", ctypes.c_int32), ("mask_kind", ctypes.c_int32),
        ("mask_rank", ctypes.c_int32), ("mask_shape", ctypes.c_int64 * 8), ("mask_strides", ctypes.c_int64 * 8),
        ("mask_row_stride", ctypes.c_int64), ("mask_col_stride", ctypes.c_int64)]


class Plan(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int32) for n in ("decode", "waves", "keys", "splits")] + [
        ("workspace_bytes", ctypes.c_size_t)]


ANY = ctypes.c_size_t(-1).value


def plan(batch, rows, cols, features, causal=False, mask=0, limit=ANY, per_call=False):
    out = Plan()
    desc = Desc(batch=batch, rows=rows, cols=cols, features=features, causal=int(causal), mask_kind=mask)
    capi.check(capi.lib().tcx_hip_flash_attention_plan(ctypes.byref(desc), ctypes.c_size_t(limit), int(per_call),
                                                       ctypes.byref(out)), "plan")
    return out


def test_no_plan_without_a_fused_kernel():
    assert capi.lib().tcx_hip_flash_attention_plan(None, 0, 0, ctypes.byref(Plan())) == capi.TCX_INVALID_ARGUMENT
    for shape in ((0, 4, 4, 64), (1, 0, 4, 64), (1, 4, -1, 64), (1, 4, 4, 20)):
        with pytest.raises(capi.HipError):
            plan(*shape)


@pytest.mark.parametrize("batch,rows,cols,features", [(4, 256, 256, 64), (16, 512, 512, 32), (2, 64, 4096, 128), (32, 1, 4096, 128),
                                                      (3, 17, 1000, 80), (8, 1024, 1024, 64)])
@pytest.mark.parametrize("causal", [False, True])
def test_split_as_far_as_the_workspace_goes(batch, rows, cols, features, causal):
    """No more splits than the workspace has room for; without one, the form
    that is best for whole rows of keys, which is the one of a call that no
    split would help."""
    full = plan(batch, rows, cols, features, causal)
    assert (full.workspace_bytes > 0) == (full.splits > 1)
    assert full.workspace_bytes == (full.splits > 1) * full.splits * batch * rows * (features + 2) * 4
    for share in (2, 3, 10):
        part = plan(batch, rows, cols, features, causal, limit=full.workspace_bytes // share)
        assert part.workspace_bytes <= full.workspace_bytes // share and part.splits <= full.splits
    none = plan(batch, rows, cols, features, causal, limit=0)
    assert (none.splits, none.workspace_bytes) == (1, 0)


def test_form_without_a_workspace():
    """Calls that no split helps take the same form with a workspace at hand and
    without; calls that are split are planned anew without one."""
    assert plan(40, 500, 500, 128).waves == plan(40, 500, 500, 128, limit=0).waves == 8
    assert plan(8, 128, 4096, 128).splits > 1
    whole, few = plan(8, 128, 4096, 128, limit=0), plan(8, 128, 128, 128, limit=0)
    assert (whole.waves, whole.keys) == (few.waves, few.keys) == (4, 32)
    assert plan(2, 64, 2048, 64).splits > 1 and plan(2, 64, 2048, 64, limit=0).keys == 64


@pytest.mark.parametrize("rows", [1, 5, 40, 64, 200])
@pytest.mark.parametrize("features", [32, 64, 80, 128])
@pytest.mark.parametrize("mask", [0, 1])
def test_causal_plans_for_the_visible_keys(rows, features, mask):
    """Keys after the last query are not run: they call for no split and no
    longer tiles (4 x 1 x 2651 x 32 was split over blocks without a key)."""
    visible, all_keys = plan(8, rows, rows, features, True, mask), plan(8, rows, 8000, features, True, mask)
    assert all_keys.splits == visible.splits and all_keys.workspace_bytes == visible.workspace_bytes
    assert rows > 64 or all_keys.splits == 1


@pytest.mark.parametrize("batch,rows,features,causal", [(8, 128, 128, True), (16, 256, 64, True), (16, 512, 32, False)])
def test_allocation_of_the_workspace_counts(batch, rows, features, causal):
    """A workspace that is allocated for the call costs 25 us from 2 MiB on,
    which these splits do not bring; in a pool that keeps it, nothing."""
    kept, once = (plan(batch, rows, rows, features, causal, per_call=c) for c in (False, True))
    assert kept.workspace_bytes >= 2 << 20 and kept.splits > 1
    assert once.workspace_bytes < 2 << 20
    long = plan(1, 64, 8192, 128, per_call=True)
    assert long.splits > 1  # 700 us of one block's keys pay for it

    fails = capi.PoolRuntime(capi.ALLOCATE_FN(lambda out, n: 1), capi.FREE_FN(lambda ptr: 0), capi.CLEAR_FN(lambda: 0))
    pool = ctypes.c_void_p()
    for limit, expected in ((1 << 30, kept), (kept.workspace_bytes, kept), (1 << 20, once)):
        capi.check(capi.lib().tcx_hip_pool_create(limit, 8, ctypes.byref(fails), ctypes.byref(pool)), "pool")
        capi.check(capi.lib().tcx_hip_pool_enter(pool), "enter")
        try:
            assert plan(batch, rows, rows, features, causal, per_call=True).splits == expected.splits
        finally:
            capi.check(capi.lib().tcx_hip_pool_exit(pool), "exit")
            capi.lib().tcx_hip_pool_destroy(pool)


# (batch, rows, cols, features, causal, waves, keys), measured both ways.
@pytest.mark.parametrize("shape", [
    (512, 100, 333, 32, False, 4, 32),    # 35.7 us; 64-key tiles 38.5 (333 keys fill 5.2 of them)
    (64, 200, 200, 32, False, 4, 64),     # one block a CU
    (512, 512, 512, 64, False, 4, 32),    # 294 us; 64-key tiles 314
    (64, 512, 512, 64, False, 4, 64),     # 45.0 us; 32-key tiles 47.2
    (300, 200, 200, 64, True, 4, 32),
    (8, 16, 1000, 32, False, 4, 64),      # one wave a block where blocks share CUs
    (512, 16, 512, 128, False, 1, 32),
    (128, 200, 8000, 64, True, 4, 32),    # the keys behind the mask are most of the work
    (32, 1000, 1000, 128, False, 8, 64),
    (64, 300, 300, 128, False, 8, 64),
    (40, 500, 500, 128, False, 8, 64),
    (32, 970, 1025, 128, False, 8, 64),
])
def test_forms(shape):
    p = plan(*shape[:5], limit=0)
    assert (p.decode, p.waves, p.keys) == (0, *shape[5:])


@pytest.mark.parametrize("rows,cols,features,mask,decode", [
    (1, 64, 32, 0, 0), (1, 65, 32, 0, 1), (2, 128, 32, 0, 0), (4, 128, 32, 0, 0), (4, 129, 32, 0, 1), (4, 16, 32, 1, 1),
    (4, 16, 64, 0, 1), (1, 1, 128, 0, 1), (4, 16, 24, 0, 1), (5, 500, 32, 0, 0), (3, 0, 64, 0, 0)])
def test_few_queries_and_keys(rows, cols, features, mask, decode):
    assert plan(300, rows, cols, features, mask=mask).decode == decode
