"""A hash-aggregate table's groups ordered and split into columns on the
device (the result of every group-by): against a sort at the sizes where
the one-block form, the sort's tiles and its digit passes end."""

import ctypes as C

import numpy as np
import pytest

from gpudbmetalcodegen_amd import _native as N
from gpudbmetalcodegen_amd import queries as Q
from helpers import group_rows

pytestmark = pytest.mark.gpu


def _check(ctx, keys, slots, variant="global"):
    r = np.random.default_rng(len(keys))
    keys = r.permutation(np.concatenate([keys, keys[: len(keys) // 3]])).astype(np.int64)
    G = {"g_key": keys.astype(np.uint32).view(np.int32), "g_val": r.integers(-10**12, 10**12, keys.size)}
    dev = Q.upload_tables(ctx, {"G": G})
    try:
        run = Q.run_groupby(ctx, dev, slots=slots, variant=variant, lds_slots=1024)
        for c, e in group_rows(G).items():
            assert run.result.columns[c].dtype == np.int64
            assert np.array_equal(run.result.columns[c], e), c
        again = run.executor.collect(run.plan)     # the workspaces and the pinned block are used again
        assert all(np.array_equal(again.columns[c], run.result.columns[c]) for c in again.columns)
    finally:
        dev["G"].free(ctx)


# groups around the one-block form's 8,192 rows (16,384 slots) and the sort's 4,096-pair tiles
@pytest.mark.parametrize("groups,slots", [(1, 64), (63, 128), (700, 2048), (4096, 8192), (8192, 16384), (8193, 16384),
                                          (12_000, 16384), (100, 32768), (4095, 65536), (4097, 65536), (70_001, 1 << 18)])
def test_groups_in_key_order(ctx, groups, slots):
    print(groups, slots, flush=True)
    _check(ctx, np.arange(1, groups + 1) * 3 + 7, slots)


# largest keys that need one to four 8-bit passes, and the ends of the key range
@pytest.mark.parametrize("top", [200, 40_000, 9_000_000, 2**31 - 1, 2**32 - 2])
def test_key_ranges(ctx, top):
    print(top, flush=True)
    r = np.random.default_rng(top)
    keys = np.unique(np.concatenate([[0, top], r.integers(0, top, 20_000)]))
    _check(ctx, keys, 1 << 16)


# the general path's result lives in page-locked memory of the runner; the one-block form's is copied
@pytest.mark.parametrize("n,slots", [(600_000, 1_200_000), (5000, 16384)])
def test_result_is_held_apart_from_the_next(ctx, n, slots):
    """A result that is still open keeps its values while the same runner
    collects others, is released and is closed."""
    eng = N.load()[1]
    G = {"g_key": np.random.default_rng(3).permutation(n).astype(np.int32), "g_val": np.arange(n, dtype=np.int64)}
    exp = group_rows(G)
    dev = Q.upload_tables(ctx, {"G": G})

    def read(r):
        rows, cols = C.c_uint64(), C.c_int()
        N.eng_check(eng.gdb_result_shape(r, C.byref(rows), C.byref(cols)))
        out = np.zeros((cols.value, rows.value), np.int64)
        N.eng_check(eng.gdb_result_words(r, out.ctypes.data))
        return out

    part = dict(variant="part", lds_slots=1024) if slots >= 65536 else dict(variant="global")
    try:
        a = Q.run_groupby(ctx, dev, slots=slots, **part)
        held = []
        for _ in range(2):
            held.append(C.c_void_p())
            N.eng_check(eng.gdb_executor_collect(a.executor.handle, a.plan.handle, C.byref(held[-1])))
        b = Q.run_groupby(ctx, dev, slots=slots, val_cut=1000, executor=a.executor, **part)
        assert b.result.rows() == 1000
        a.executor.release()
        a.executor.close()
        for r in held:
            for got, e in zip(read(r), exp.values()):
                assert np.array_equal(got, e)
            N.eng_check(eng.gdb_result_free(r))
    finally:
        dev["G"].free(ctx)
