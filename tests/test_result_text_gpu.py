"""A collected result against itself: the canonical CSV rendered again in
Python from the columns and formats, over results with fixed-point, 128-bit,
negative, date and string columns, extreme values, no rows, and labels that
hold the separators of the one-call description."""

import ctypes as C

import numpy as np
import pytest

from gpudbmetalcodegen_amd import _native as N
from gpudbmetalcodegen_amd import queries as Q
from gpudbmetalcodegen_amd import tpch as T
from gpudbmetalcodegen_amd import tpch_gen as G
from gpudbmetalcodegen_amd import workloads as W

pytestmark = pytest.mark.gpu


def _text(res) -> str:
    lines = [",".join(res.columns)]
    for r in range(res.rows()):
        f = []
        for name, col in res.columns.items():
            scale, date = res.formats[name]
            v = col[r]
            if isinstance(v, str):
                f.append('"' + v.replace('"', '""') + '"' if any(c in v for c in ',"\n\r') else v)
            elif date:
                f.append(f"{int(v) // 10000:04d}-{int(v) // 100 % 100:02d}-{int(v) % 100:02d}")
            elif scale:
                d = str(abs(int(v))).rjust(scale + 1, "0")
                f.append(("-" if v < 0 else "") + d[:-scale] + "." + d[-scale:])
            else:
                f.append(str(int(v)))
        lines.append(",".join(f))
    return "\n".join(lines) + "\n"


def test_named_plans_text(ctx):
    db = T.TpchDB(ctx, G.generate(0.01, seed=3))
    try:
        for q in ("Q1", "Q3", "Q6", "Q10", "Q11", "Q13", "Q18", "Q21", "Q22"):
            res = T.run(ctx, db, q).raw
            assert res.canonical == _text(res), q
        for label in ("M\x1fA", "M\x1eA", 'M"A'):
            r = T.run(ctx, db, "Q12", options=f"mode1={label}")
            assert r.raw.canonical == _text(r.raw) and label in list(next(iter(r.raw.columns.values())))
    finally:
        db.free()


@pytest.mark.parametrize("bins", [5, 4095, 4096, 4097, 9000])
def test_counts_around_the_largest_piece(ctx, bins):
    """Histograms read with the run's other words, and beyond 16 KB by a copy."""
    db = T.TpchDB(ctx, G.generate(0.01, seed=3))
    try:
        res, exp = T.run(ctx, db, "Q13", options=f"hist_bins={bins}").raw, T.run(ctx, db, "Q13").raw
        rows = [(c, n) for c, n in zip(exp.columns["c_count"], exp.columns["custdist"]) if c < bins]
        assert list(zip(res.columns["c_count"], res.columns["custdist"])) == rows and res.canonical == _text(res)
    finally:
        db.free()


def test_scan_text_and_no_rows(ctx):
    dev = Q.upload_tables(ctx, W.workload0(5000))
    try:
        for cutoff in (W.q1_cutoff(), -1):
            res = Q.run_q1(ctx, dev, cutoff).result
            assert res.canonical == _text(res) and res.rows() == (6 if cutoff >= 0 else 0)
            assert all(v.dtype == (np.int64 if k.startswith(("sum_qty", "sum_base", "count")) else v.dtype)
                       for k, v in res.columns.items())
    finally:
        dev["F"].free(ctx)


def test_extreme_values_text(ctx):
    lo, hi = -2**63, 2**63 - 1
    G_ = {"g_key": np.array([1, 2, 3, 4, 4], np.int32), "g_val": np.array([lo, hi, 0, -1, 1], np.int64)}
    dev = Q.upload_tables(ctx, {"G": G_})
    try:
        res = Q.run_groupby(ctx, dev, slots=64, variant="global").result
        assert list(res.columns["min"]) == [lo, hi, 0, -1] and list(res.columns["max"]) == [lo, hi, 0, 1]
        assert res.canonical == _text(res)
    finally:
        dev["G"].free(ctx)


def test_column_calls_refuse_other_columns(ctx):
    """Indexes outside the result and columns of another type are errors."""
    dev = Q.upload_tables(ctx, W.workload0(5000))
    eng, r = N.load()[1], C.c_void_p()
    try:
        run = Q.run_q1(ctx, dev, W.q1_cutoff())
        N.eng_check(eng.gdb_executor_collect(run.executor.handle, run.plan.handle, C.byref(r)))
        rows, cols = run.result.rows(), len(run.result.columns)
        out = np.zeros(2 * rows, np.int64)
        types = []
        for i in range(cols):
            got = (eng.gdb_result_i64(r, i, out.ctypes.data), eng.gdb_result_i128(r, i, out.ctypes.data),
                   eng.gdb_result_str(r, i, C.create_string_buffer(64 * rows), 64))
            assert sorted(got) == [N.GDB_OK, N.GDB_ERR_INVALID, N.GDB_ERR_INVALID]
            types.append(got.index(N.GDB_OK))
        assert set(types) == {0, 1, 2}
        for i in (-1, cols):
            for st in (eng.gdb_result_i64(r, i, None), eng.gdb_result_i128(r, i, None), eng.gdb_result_str(r, i, None, 64)):
                assert st == N.GDB_ERR_INVALID and b"index out of range" in eng.gdb_engine_last_error()
        N.eng_check(eng.gdb_result_free(r))
    finally:
        dev["F"].free(ctx)
