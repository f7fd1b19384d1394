"""Top-10 over per-block candidate lists and the queued hash build of the
join: fewer result rows than K, one block and many, blocks of fewer threads
than lists, ties in the rank's first word, every row passing and none. Exact
against the oracle."""

import ctypes as C

import numpy as np
import pytest

import oracle
from gpudbmetalcodegen_amd import _native as N
from gpudbmetalcodegen_amd import queries as Q
from tests.test_oracle import small_join

pytestmark = pytest.mark.gpu


def _run(ctx, A, B, F, seg, d, options):
    dev = Q.upload_tables(ctx, {"A": A, "B": B, "F": F})
    try:
        run = Q.run_q3(ctx, dev, seg, d, options, int(A["a_key"].max()), int(B["b_key"].max()))
        top = {k: [int(x) for x in v] for k, v in run.result.columns.items()}
        assert top == {k: v.tolist() for k, v in oracle.q3_topk(A, B, F, seg, d, 10).items()}
        groups, exp = Q.q3_hash_groups(run), oracle.q3(A, B, F, seg, d)
        for c in ("key", "rev", "date"):
            assert np.array_equal(groups[c], exp[c]), c
        return run.result.rows()
    finally:
        for t in dev.values():
            t.free(ctx)


@pytest.mark.parametrize("options", ["", "merge_block=64", "merge_block=1024", "items_topk=16", "compact_b=0",
                                     "items_b=8", "block_b=1024,items_b=8", "bflags=1"])
@pytest.mark.parametrize("n_b", [1, 63, 65, 2049, 120_001])
def test_topk_and_queued_build(ctx, n_b, options):
    A, B, F = small_join(20 + n_b % 7, n_a=max(1, n_b // 10), n_b=n_b)
    A["a_seg"][:] = 2                          # every B row passes the bitmap
    assert _run(ctx, A, B, F, 2, 60, options) <= 10


@pytest.mark.parametrize("options", ["", "merge_block=64"])
def test_topk_equal_revenue(ctx, options):
    A, B, F = small_join(31, n_a=500, n_b=30_000)
    A["a_seg"][:] = 2
    F["f_price"][:] = 700
    F["f_disc"][:] = 5                         # revenue ties; date and key decide
    _run(ctx, A, B, F, 2, 60, options)


@pytest.mark.parametrize("block", [64, 1024])
def test_queued_build_at_other_blocks(ctx, block):
    """Blocks below and above the default of a compiled plan."""
    A, B, F = small_join(41, n_a=5000, n_b=50_003)
    A["a_seg"][:] = 2
    plan = Q.get_plan(ctx, "Q3", "")
    shape = plan.get_launch("Q3_build_b_table")
    plan.set_launch("Q3_build_b_table", block, shape[1])
    try:
        _run(ctx, A, B, F, 2, 60, "")
    finally:
        plan.set_launch("Q3_build_b_table", *shape)
    _run(ctx, A, B, F, 2, 60, "")


def test_autotuned_queued_build(ctx):
    A, B, F = small_join(42, n_a=5000, n_b=50_003)
    dev = Q.upload_tables(ctx, {"A": A, "B": B, "F": F})
    try:
        run = Q.run_q3(ctx, dev, 2, 60, "", int(A["a_key"].max()), int(B["b_key"].max()))
        plan, text = run.plan, run.result.canonical
        shape = plan.get_launch("Q3_build_b_table")
        bl, it = (C.c_int * 3)(1024, 256, 512), (C.c_int * 1)(shape[1])
        block, n, ms, count, table = C.c_int(), C.c_int(), C.c_float(), C.c_int(), (C.c_double * 12)()
        N.eng_check(N.load()[1].gdb_autotune_phase(run.executor.handle, plan.handle, b"Q3_build_b_table", bl, 3, it, 1,
                                                   None, None, 0, 2, C.byref(block), C.byref(n), None, C.byref(ms), table,
                                                   C.byref(count)))
        try:
            assert count.value == 3 and sorted(table[0::4]) == [256, 512, 1024] and ms.value == pytest.approx(min(table[3::4]))
            assert plan.get_launch("Q3_build_b_table") == (block.value, shape[1])
            run.executor.execute(plan)
            assert run.executor.collect(plan).canonical == text
        finally:
            plan.set_launch("Q3_build_b_table", *shape)
    finally:
        for t in dev.values():
            t.free(ctx)
