"""Several runners' results read together equal the same results read one by
one: group tables in one launch and two, tables that need the general path,
scalar and top-k results, another stream, the same runner twice, none."""

import ctypes as C

import numpy as np
import pytest

from gpudbmetalcodegen_amd import _native as N
from gpudbmetalcodegen_amd import engine as E
from gpudbmetalcodegen_amd import queries as Q
from gpudbmetalcodegen_amd import workloads as W
from tests.test_oracle import small_join

pytestmark = pytest.mark.gpu


def _groups(ctx, n, slots, stream=None):
    r = np.random.default_rng(n + slots)
    rows = max(n, 100)
    G = {"g_key": r.permutation(np.arange(rows, dtype=np.int32) * 5 + 1), "g_val": r.integers(-10**9, 10**9, rows)}
    dev = Q.upload_tables(ctx, {"G": G})
    cut = None if n == rows else int(np.sort(G["g_val"])[n])   # n rows pass
    run = Q.run_groupby(ctx, dev, slots=slots, variant="global", val_cut=cut, executor=E.HipGenericExecutor(ctx, stream))
    assert run.result.rows() == n
    return run, dev


# no runner, 0 groups (every row cut) in the one-block form and the general path, the one-block form's ends, the
# general path, and 70 tables (two launches)
@pytest.mark.parametrize("sizes", [[], [(0, 64), (5, 64), (0, 65536)], [(1, 64)], [(700, 2048)] * 3, [(8192, 16384), (8193, 16384), (20_000, 65536), (63, 128)],
                                   [(10 + i, 64 + 64 * (i % 2)) for i in range(70)]])
def test_group_tables(ctx, sizes):
    made = [_groups(ctx, n, slots) for n, slots in sizes]
    try:
        runs = [(r.executor, r.plan) for r, _ in made]
        got = E.HipGenericExecutor.collect_many(runs + runs[:1])
        assert len(got) == len(runs) + min(1, len(runs))
        for g, (r, _) in zip(got, made + made[:1]):
            assert g.canonical == r.result.canonical
            assert all(np.array_equal(g.columns[c], r.result.columns[c]) for c in r.result.columns)
    finally:
        for r, dev in made:
            r.executor.close()
            dev["G"].free(ctx)


def test_mixed_results_and_streams(ctx):
    F = W.fact_f(5000, 3)
    A, B, J = small_join(5)
    fdev, jdev = Q.upload_tables(ctx, {"F": F}), Q.upload_tables(ctx, {"A": A, "B": B, "F": J})
    (hip, _), st = N.load(), C.c_void_p()
    N.hip_check(hip.gdb_stream_create(ctx.handle, C.byref(st)))
    made = [_groups(ctx, 300, 1024), _groups(ctx, 500, 1024, st)]
    try:
        scans = [Q.run_q1(ctx, fdev, c, executor=E.HipGenericExecutor(ctx)) for c in (0, W.q1_cutoff(), 900)] * 20
        join = Q.run_q3(ctx, jdev, 2, 50, "", int(A["a_key"].max()), int(B["b_key"].max()),
                        executor=E.HipGenericExecutor(ctx))
        all_runs = [made[0][0], *scans, join, made[1][0]]
        got = E.HipGenericExecutor.collect_many([(r.executor, r.plan) for r in all_runs])
        for g, r in zip(got, all_runs):
            assert g.canonical == r.result.canonical
    finally:
        made[1][0].executor.close()
        N.hip_check(hip.gdb_stream_destroy(st))
        for t in (*fdev.values(), *jdev.values(), made[0][1]["G"], made[1][1]["G"]):
            t.free(ctx)
