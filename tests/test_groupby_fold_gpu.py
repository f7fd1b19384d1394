"""The LDS group-by's fold phase (partial tables -> group table): against a
sort where it can go wrong — few blocks (no partials), LDS tables smaller
than the groups (spills, keys probing past their home slot and round the
table's end), tables filled over several runs or chunks, and as work items of
a batch; and the fold's launch shape tuned."""

import ctypes as C

import numpy as np
import pytest

from gpudbmetalcodegen_amd import _native as N
from gpudbmetalcodegen_amd import batch as B
from gpudbmetalcodegen_amd import engine as E
from gpudbmetalcodegen_amd import queries as Q
from helpers import group_rows

pytestmark = pytest.mark.gpu


def _table(n, groups, seed, skew=False):
    r = np.random.default_rng(seed)
    k = r.integers(0, groups, n) if not skew else np.minimum(r.zipf(1.3, n), groups) - 1
    return {"g_key": ((k * 2654435761) % (1 << 31)).astype(np.int32), "g_val": r.integers(-10**9, 10**9, n)}


def _same(cols, G, times=1):
    for c, e in group_rows(G).items():
        assert np.array_equal(cols[c], e * (times if c in ("count", "sum") else 1)), c


# rows: below and above 16 blocks of 2,048; groups: far below, at and above the LDS slots
@pytest.mark.parametrize("lds_slots", [64, 1024, 4096])
@pytest.mark.parametrize("n,groups", [(1, 1), (30_000, 500), (40_000, 500), (300_001, 60), (300_001, 1000), (300_001, 5000)])
@pytest.mark.parametrize("skew", [False, True])
def test_fold_matches_oracle(ctx, lds_slots, n, groups, skew):
    print(lds_slots, n, groups, skew, flush=True)
    G = _table(n, groups, n + lds_slots, skew)
    dev = Q.upload_tables(ctx, {"G": G})
    try:
        run = Q.run_groupby(ctx, dev, slots=2 * groups, variant="lds", lds_slots=lds_slots)
        _same(run.result.columns, G)
        run.executor.execute(run.plan, 1, 2)
        _same(run.executor.collect(run.plan).columns, G)
        # two runs into one table: the second folds only its own partials
        run.executor.execute(run.plan)
        run.executor.set_skip_init(True)
        run.executor.execute(run.plan)
        _same(run.executor.collect(run.plan).columns, G, times=2)
    finally:
        dev["G"].free(ctx)


def test_partial_tables_take_the_room_the_rows_need(ctx):
    """A small table's runner holds little; the same runner then serves a larger
    table, and again the small one."""
    small, large = _table(1000, 300, 3), _table(300_001, 900, 4)
    dev = Q.upload_tables(ctx, {"G": small}), Q.upload_tables(ctx, {"G": large})
    try:
        run = Q.run_groupby(ctx, dev[0], slots=2048, variant="lds")
        _same(run.result.columns, small)
        assert run.executor.owned_bytes() < 1 << 20
        for k, G in ((1, large), (0, small)):
            again = Q.run_groupby(ctx, dev[k], slots=2048, variant="lds", executor=run.executor)
            _same(again.result.columns, G)
    finally:
        for d in dev:
            d["G"].free(ctx)


# blocks of 4,096 rows against room for 512 partials (lds_slots 2048) or 256 (4096): several chunks' partials,
# chunks of too few blocks to leave any, one chunk, and more partials than there is room for
@pytest.mark.parametrize("n,chunk,lds_slots", [(500_000, 100_000, 2048), (500_000, 4096, 2048), (500_000, 500_000, 2048),
                                               (1_400_000, 100_000, 4096)])
def test_fold_of_a_chunked_run(ctx, n, chunk, lds_slots):
    G = _table(n, 700, 5)
    h = E.HostTable("G", G)
    try:
        run = Q.run_groupby(ctx, {}, slots=2048, variant="lds", lds_slots=lds_slots, stream=Q.Stream(h, chunk))
        _same(run.result.columns, G)
    finally:
        h.close()


# 1, 3 partials for some 100 blocks a pipeline: the other blocks merge directly
@pytest.mark.parametrize("partials", [1, 3])
def test_more_blocks_than_partials(ctx, partials):
    w = B.Workload3(ctx, B.workload3(n_pipes=8, scale=0.2, seed=79), lds_cap=4096, partials=partials)
    try:
        w.run_plain()
        plain = w.results()
        aggs = [s.index for s in w.specs if s.kind == "agg"]
        blocks = []
        for i in aggs:
            blocks.append(w.execs[i].execute(w.batch_plans["agg"]).phases[0][2])
            got = w.execs[i].collect(w.batch_plans["agg"]).columns
            assert all(np.array_equal(got[k], plain[i][k]) for k in plain[i]), i
        assert max(blocks) > 16
        b = w.build_batch(512, 16_384)   # several work items a pipeline
        try:
            for _ in range(2):
                b.run(graph=True)
                for got, exp in zip(w.results(), plain):
                    assert all(np.array_equal(got[k], exp[k]) for k in exp)
        finally:
            b.close()
    finally:
        w.close()


@pytest.mark.parametrize("chunk", [2048, 20_000, 1 << 20])
@pytest.mark.parametrize("lds_bits", [5, 9, 12])
def test_fold_of_batched_pipelines(ctx, chunk, lds_bits):
    specs = B.workload3(n_pipes=8, scale=0.05, seed=77)
    w = B.Workload3(ctx, specs, lds_cap=4096, partials=32)
    try:
        w.run_plain()
        plain = w.results()
        for s in w.specs:
            w.batch_launch[s.index] = (256, 4, lds_bits)
        b = w.build_batch(512, 16_384, fold_rows=chunk)
        try:
            for _ in range(3):
                b.run(graph=True)
                for got, exp in zip(w.results(), plain):
                    assert all(np.array_equal(got[k], exp[k]) for k in exp)
        finally:
            b.close()
    finally:
        w.close()


def test_scan_phase_alone_leaves_the_whole_table(ctx):
    """Phase ranges: the scan without its fold, the fold after it on its own,
    and both together hold every group once."""
    G = _table(300_001, 900, 7)
    dev = Q.upload_tables(ctx, {"G": G})
    try:
        run = Q.run_groupby(ctx, dev, slots=2048, variant="lds")
        ex, plan = run.executor, run.plan
        assert plan.phases() == ["GB_agg", "GB_merge"]
        ex.execute(plan, first=0, last=1)
        _same(ex.collect(plan).columns, G)
        ex.execute(plan, first=1, last=2)
        _same(ex.collect(plan).columns, G)
        ex.execute(plan)
        _same(ex.collect(plan).columns, G)
    finally:
        dev["G"].free(ctx)


def test_pipeline_scan_alone_leaves_the_whole_table(ctx):
    w = B.Workload3(ctx, B.workload3(n_pipes=8, scale=0.2, seed=78), lds_cap=4096, partials=32)
    try:
        w.run_plain()
        plain = w.results()
        for s in w.specs:
            if s.kind == "agg":
                w.execs[s.index].execute(w.batch_plans["agg"], first=0, last=1)
        for got, exp in zip(w.results(), plain):
            assert all(np.array_equal(got[k], exp[k]) for k in exp)
    finally:
        w.close()


def _autotune(ex, plan, phase, blocks, items):
    bl, it = (C.c_int * len(blocks))(*blocks), (C.c_int * len(items))(*items)
    block, n, ms, count = C.c_int(), C.c_int(), C.c_float(), C.c_int()
    table = (C.c_double * (4 * len(blocks) * len(items)))()
    N.eng_check(N.load()[1].gdb_autotune_phase(ex.handle, plan.handle, phase.encode(), bl, len(blocks), it, len(items),
                                               None, None, 0, 3, C.byref(block), C.byref(n), None, C.byref(ms), table,
                                               C.byref(count)))
    assert block.value in blocks and ms.value > 0
    return count.value


@pytest.mark.parametrize("phase", ["GB_agg", "GB_merge"])
def test_autotuned_fold_folds_in_every_trial(ctx, phase):
    """Each trial fills and folds partials: after tuning, the group table holds
    the rows of the table registered by then, not those of the run before."""
    first, second = _table(300_001, 900, 1), _table(300_001, 400, 2)
    dev = Q.upload_tables(ctx, {"G": first})
    other = Q.upload_tables(ctx, {"G": second})
    try:
        run = Q.run_groupby(ctx, dev, slots=2048, variant="lds")
        _same(run.result.columns, first)
        shape = run.plan.get_launch(phase)
        run.executor.register_table(other["G"])
        assert _autotune(run.executor, run.plan, phase, (64, 256, 1024), [shape[1]]) == 3
        _same(run.executor.collect(run.plan).columns, second)
        run.plan.set_launch(phase, *shape)
    finally:
        dev["G"].free(ctx)
        other["G"].free(ctx)
