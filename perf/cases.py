"""Performance cases of the query engine: what a program that uses it has it do,
called through the query drivers (``queries``, ``estimator``, ``batch``,
``tpch``, ``sql``) with tables resident in HBM, from the smallest calls, where
latency and launches count, to the full shapes of the benchmark.

A case is a dict of plain values; ``case["kind"]`` names the driver:

  scan     fused filter + small group-by (TPC-H Q1 shape): ``queries.run_q1``
  join     semi-join bitmap, hash build, probe, top-10: ``queries.run_q3``
  group    hash group-by, sized exactly or by the estimator:
           ``queries.run_groupby`` / ``estimator.run_groupby_learned``
  like     LIKE '%w1%w2%' + per-key count + histogram: ``queries.run_q13``
  anti     bitmap anti-join + per-segment aggregate: ``queries.run_q22``
  batch    many uneven pipelines in one graph replay: ``batch.Workload3``
  tpch     named TPC-H plans: ``tpch.run``
  sql      TPC-H queries planned from their text: ``sql.run_sql``

A pass is one call with its results on the host, as a program that asked the
question needs them. Every result is whole numbers, so outputs compare exactly.
"""

from __future__ import annotations

import math
from pathlib import Path

import numpy as np
import torch

from gpudbmetalcodegen_amd import batch as B
from gpudbmetalcodegen_amd import engine as E
from gpudbmetalcodegen_amd import estimator as EST
from gpudbmetalcodegen_amd import queries as Q
from gpudbmetalcodegen_amd import sql as S
from gpudbmetalcodegen_amd import tpch as T
from gpudbmetalcodegen_amd import workloads as W

PKG = Path(E.__file__).resolve().parent

# SQL text as a program sends it (TPC-H Q1, Q6 and Q12)
SQL = {
    "Q1": "select l_returnflag, l_linestatus, sum(l_quantity) as sum_qty, sum(l_extendedprice) as sum_base_price, "
          "sum(l_extendedprice * (1 - l_discount)) as sum_disc_price, "
          "sum(l_extendedprice * (1 - l_discount) * (1 + l_tax)) as sum_charge, avg(l_quantity) as avg_qty, "
          "avg(l_extendedprice) as avg_price, avg(l_discount) as avg_disc, count(*) as count_order "
          "from lineitem where l_shipdate <= date '1998-12-01' - interval '90' day "
          "group by l_returnflag, l_linestatus order by l_returnflag, l_linestatus",
    "Q6": "select sum(l_extendedprice * l_discount) as revenue from lineitem where l_shipdate >= date '1994-01-01' "
          "and l_shipdate < date '1994-01-01' + interval '1' year "
          "and l_discount between .06 - 0.01 and .06 + 0.01 and l_quantity < 24",
    "Q12": "select l_shipmode, "
           "sum(case when o_orderpriority = '1-URGENT' or o_orderpriority = '2-HIGH' then 1 else 0 end) as high_line_count, "
           "sum(case when o_orderpriority <> '1-URGENT' and o_orderpriority <> '2-HIGH' then 1 else 0 end) as low_line_count "
           "from orders, lineitem where o_orderkey = l_orderkey and l_shipmode in ('MAIL', 'SHIP') "
           "and l_commitdate < l_receiptdate and l_shipdate < l_commitdate and l_receiptdate >= date '1994-01-01' "
           "and l_receiptdate < date '1994-01-01' + interval '1' year group by l_shipmode order by l_shipmode",
}


def listed():
    return [
        # an interactive dashboard's query on a small table: nothing but latency
        {"name": "scan_10k", "kind": "scan", "rows": 10_000, "cutoff": 2435},
        # the fused scan-aggregate at the full fact table
        {"name": "scan_120m", "kind": "scan", "rows": 120_000_000, "cutoff": 2435},
        # a join of small, odd-sized tables
        {"name": "join_600k", "kind": "join", "a": 15_013, "b": 150_001, "seg": 2, "date": 1203},
        # the three-way join + top-10 at the benchmark's shape (about 60M fact rows)
        {"name": "join_60m", "kind": "join", "a": 1_500_000, "b": 15_000_000, "seg": 2, "date": 1203},
        # few groups: the LDS table holds them all; the result is a few hundred rows
        {"name": "group_few_1m", "kind": "group", "rows": 1_000_003, "groups": 700, "skew": 0.0, "variant": "lds",
         "cut": 0, "sizing": "prepass"},
        # many skewed groups (a third of the benchmark's shape), sized by the exact pre-pass
        {"name": "group_zipf_40m", "kind": "group", "rows": 40_000_000, "groups": 2_200_000, "skew": 1.1,
         "variant": "part", "cut": 0, "sizing": "prepass"},
        # filtered group-by over near-uniform keys, table sized by the estimator
        {"name": "group_learned_8m", "kind": "group", "rows": 8_000_000, "groups": 400_000, "skew": 0.5,
         "variant": "part", "cut": 500_000, "sizing": "learned"},
        # byte-exact LIKE over the served string table
        {"name": "like_4m", "kind": "like", "rows": 4_000_000, "a": 3_000_000, "negate": False},
        # anti-join of the served tables
        {"name": "anti_30m", "kind": "anti", "b": 30_000_000, "a": 3_000_000, "lo": 700, "hi": 950},
        # 64 pipelines of 10^4..10^7 rows in one graph replay
        {"name": "batch_64", "kind": "batch", "pipes": 64, "scale": 1.0},
        # the named TPC-H queries the reference publishes times for, SF 1
        {"name": "tpch_sf1", "kind": "tpch", "sf": 1.0, "queries": "Q1 Q4 Q6 Q13 Q22"},
        # queries sent as text, SF 0.2
        {"name": "sql_sf02", "kind": "sql", "sf": 0.2, "queries": "Q1 Q6 Q12"},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm, odd ones among them."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["scan", "scan", "join", "join", "group", "group", "group", "like", "anti", "batch", "tpch", "sql"])
    if kind == "scan":
        return {"kind": kind, "rows": _log(rng, 3_000, 120_000_000), "cutoff": rng.randint(100, 2525)}
    if kind == "join":
        b = _log(rng, 20_000, 15_000_000)
        return {"kind": kind, "a": max(16, b // rng.randint(8, 20)), "b": b, "seg": rng.randint(0, 4),
                "date": rng.randint(300, 1600)}
    if kind == "group":
        rows = _log(rng, 20_000, 40_000_000)
        groups = _log(rng, 16, max(64, rows // 16))
        learned = rng.random() < 0.4
        return {"kind": kind, "rows": rows, "groups": groups, "skew": rng.choice([0.0, 0.5, 0.8, 1.1, 1.4]),
                "variant": "part" if groups > 30_000 else "lds", "cut": rng.choice([0, 0, 50_000, 500_000, 900_000]),
                "sizing": "learned" if learned else "prepass"}
    if kind == "like":
        rows = _log(rng, 5_000, 4_000_000)
        return {"kind": kind, "rows": rows, "a": max(100, rows * 3 // rng.randint(4, 12)), "negate": rng.random() < 0.5}
    if kind == "anti":
        b = _log(rng, 20_000, 30_000_000)
        lo = rng.randint(0, 2000)
        return {"kind": kind, "b": b, "a": max(100, b // rng.randint(8, 20)), "lo": lo, "hi": lo + rng.randint(50, 400)}
    if kind == "batch":
        return {"kind": kind, "pipes": 2 * rng.randint(4, 32), "scale": round(rng.uniform(0.05, 1.0), 3)}
    if kind == "tpch":
        qs = sorted(rng.sample(["Q1", "Q4", "Q6", "Q13", "Q22"], rng.randint(1, 5)), key=lambda q: int(q[1:]))
        return {"kind": kind, "sf": round(math.exp(rng.uniform(math.log(0.02), 0.0)), 3), "queries": " ".join(qs)}
    qs = rng.sample(sorted(SQL), rng.randint(1, 3))
    return {"kind": kind, "sf": round(math.exp(rng.uniform(math.log(0.01), math.log(0.2))), 3), "queries": " ".join(qs)}


# ---------------------------------------------------------------------------
# Inputs, made on the GPU (or by the engine's generators) from the seed alone
# ---------------------------------------------------------------------------

_CTX: list = []


def _ctx() -> E.Context:
    if not _CTX:
        c = E.Context(0)
        cache = PKG / "_cocache"
        if cache.exists():
            c.set_cache_dir(str(cache))
        _CTX.append(c)
    return _CTX[0]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1_000_003 + 17)


def _uniform(g, n, lo, hi, dtype):
    """n whole numbers of [lo, hi]."""
    return torch.randint(lo, hi + 1, (n,), generator=g, device="cuda", dtype=dtype)


def _permutation(g, n):
    return (torch.randperm(n, generator=g, device="cuda", dtype=torch.int32) + 1).to(torch.int32)


def _zipf(g, n, s, keys):
    """Keys 1..keys with P(k) close to k^-s (the inverse of the continuous distribution function)."""
    if s == 0.0:
        return _uniform(g, n, 1, keys, torch.int32)
    out = torch.empty(n, dtype=torch.int32, device="cuda")
    for b in range(0, n, 16_777_216):
        u = torch.rand(min(n - b, 16_777_216), generator=g, device="cuda", dtype=torch.float64)
        e = 1.0 - s
        x = (u * ((keys + 1.0) ** e - 1.0) + 1.0) ** (1.0 / e)
        out[b:b + u.numel()] = x.floor().clamp_(1, keys).to(torch.int32)
    return out


def _fact(n, seed):
    g = _gen(seed)
    flag = torch.tensor([65, 82, 78, 78], dtype=torch.uint8, device="cuda")   # A, R, N in ratio 1:1:2
    status = torch.tensor([70, 79], dtype=torch.uint8, device="cuda")         # F, O
    return {"F": {"f_qty": _uniform(g, n, 1, 50, torch.int32),
                  "f_price": _uniform(g, n, W.PRICE_LO, W.PRICE_HI, torch.int64),
                  "f_disc": _uniform(g, n, 0, 10, torch.int32), "f_tax": _uniform(g, n, 0, 8, torch.int32),
                  "f_flag": flag[_uniform(g, n, 0, 3, torch.int64)],
                  "f_status": status[_uniform(g, n, 0, 1, torch.int64)],
                  "f_date": _uniform(g, n, 0, W.DATE_DAYS_W0 - 1, torch.int32)}}


def _dims(g, n_a, n_b):
    a = {"a_key": _permutation(g, n_a), "a_seg": _uniform(g, n_a, 0, 4, torch.uint8)}
    b = {"b_key": _permutation(g, n_b), "b_fkey": _uniform(g, n_b, 1, n_a, torch.int32),
         "b_date": _uniform(g, n_b, 0, W.DATE_DAYS_W1 - 1, torch.int32)}
    return a, b


def _join_tables(n_a, n_b, seed):
    g = _gen(seed)
    a, b = _dims(g, n_a, n_b)
    per = _uniform(g, n_b, 1, 7, torch.int64)                # 1..7 fact rows per B key, in no order
    fk = torch.repeat_interleave(torch.arange(1, n_b + 1, device="cuda", dtype=torch.int32), per)
    n = fk.numel()
    fk = fk[torch.randperm(n, generator=g, device="cuda")]
    return {"A": a, "B": b, "F": {"f_fkey": fk, "f_price": _uniform(g, n, W.PRICE_LO, W.PRICE_HI, torch.int64),
                                  "f_disc": _uniform(g, n, 0, 10, torch.int32),
                                  "f_date": _uniform(g, n, 0, W.DATE_DAYS_W1 - 1, torch.int32)}}


def _group_table(n, s, groups, cut, seed):
    """n rows of `groups` keys, one in each three of 1..3 * groups: every key has a row that
    the filter keeps, the other rows follow Zipf(s); small keys are the frequent ones."""
    g = _gen(seed)
    ids = torch.arange(groups, device="cuda", dtype=torch.int32) * 3 + _uniform(g, groups, 1, 3, torch.int32)
    rank = torch.cat([torch.arange(groups, device="cuda", dtype=torch.int32), _zipf(g, n - groups, s, groups) - 1])
    val = _uniform(g, n, 0, 1_000_000, torch.int64)
    if cut:
        val[:groups] %= cut
    order = torch.randperm(n, generator=g, device="cuda")
    return {"G": {"g_key": ids[rank[order].to(torch.int64)], "g_val": val[order]}}


def _text_tables(n, n_a, seed):
    vocab = W.vocabulary(seed)
    g = _gen(seed)
    s = {"s_fkey": _uniform(g, n, 1, n_a, torch.int32),
         "s_text": torch.from_numpy(W.text(seed, 52, n, W.S_WIDTH, vocab)).cuda()}
    a = {"a_key": _permutation(g, n_a), "a_seg": _uniform(g, n_a, 0, 4, torch.uint8)}
    r = np.random.default_rng(seed)
    i, j = r.integers(0, len(vocab), 2)          # fragments short enough to occur in the smallest tables
    return {"S": s, "A": a}, vocab[i][:2], vocab[j][:1]


_DAYS = np.array([(y * 10000 + m * 100 + d) for y in range(1992, 2000) for m in range(1, 13)
                  for d in range(1, (29 if y % 4 == 0 else 28) + 1 if m == 2 else 31 if m in (4, 6, 9, 11) else 32)],
                 dtype=np.int32)


def _tpch_host(sf, seed):
    """lineitem, orders and customer at scale factor sf with TPC-H's domains: 1..7 lines
    per order in order-key sequence, dates following the order's, sparse order keys."""
    r = np.random.default_rng(seed)
    n_ord, n_cust = max(8, int(1_500_000 * sf)), max(9, int(150_000 * sf))
    i = np.arange(n_ord, dtype=np.int64)
    okey = ((i // 8) * 32 + i % 8 + 1).astype(np.int32)
    active = np.arange(1, n_cust + 1, dtype=np.int32)
    active = active[active % 3 != 0]
    oday = r.integers(0, 2406 - 151, n_ord, dtype=np.int32)
    lines = r.integers(1, 8, n_ord)
    n = int(lines.sum())
    day = np.repeat(oday, lines)
    ship = day + W.uniform_i32(seed, 1, n, 1, 121)
    receipt = ship + W.uniform_i32(seed, 2, n, 1, 30)
    commit = day + W.uniform_i32(seed, 3, n, 30, 90)
    qty = W.uniform_i64(seed, 4, n, 1, 50)
    modes = np.frombuffer(b"REAIRAMASHTRFO", np.uint8).reshape(7, 2)      # the catalog keeps two bytes
    today = int(np.searchsorted(_DAYS, 19950617))
    lineitem = {
        "l_orderkey": np.repeat(okey, lines), "l_partkey": W.uniform_i32(seed, 15, n, 1, max(1, int(200_000 * sf))),
        "l_quantity": qty * 100,
        "l_extendedprice": qty * W.uniform_i64(seed, 5, n, 90_000, 200_000),
        "l_discount": W.uniform_i64(seed, 6, n, 0, 10), "l_tax": W.uniform_i64(seed, 7, n, 0, 8),
        "l_returnflag": np.where(receipt <= today, W.categorical_u8(seed, 8, n, b"RA", [1, 1]), ord("N")).astype(np.uint8),
        "l_linestatus": np.where(ship > today, ord("O"), ord("F")).astype(np.uint8),
        "l_shipdate": _DAYS[ship], "l_commitdate": _DAYS[commit], "l_receiptdate": _DAYS[receipt],
        "l_shipmode": modes[W.uniform_i32(seed, 9, n, 0, 6)],
    }
    words = W.vocabulary(seed, 200)
    words[3], words[77] = b"special", b"requests"
    orders = {
        "o_orderkey": okey, "o_custkey": active[r.integers(0, active.size, n_ord)], "o_orderdate": _DAYS[oday],
        "o_orderpriority": W.categorical_u8(seed, 10, n_ord, b"12345", [1] * 5),
        "o_comment": W.text(seed, 11, n_ord, 79, words),
    }
    phone = W.uniform_i32(seed, 12, n_cust * 15, ord("0"), ord("9")).astype(np.uint8).reshape(n_cust, 15)
    code = W.uniform_i32(seed, 13, n_cust, 10, 34)
    phone[:, 0], phone[:, 1], phone[:, 2] = ord("0") + code // 10, ord("0") + code % 10, ord("-")
    customer = {"c_custkey": np.arange(1, n_cust + 1, dtype=np.int32), "c_phone": phone,
                "c_acctbal": W.uniform_i64(seed, 14, n_cust, -99_999, 999_999)}
    return {"lineitem": lineitem, "orders": orders, "customer": customer}


class State:
    """What the program keeps between calls: tables in HBM, runners, plans."""

    def __init__(self, case):
        self.case = case
        self.keep = []
        self.close = []

    def tables(self, cols):
        self.keep.append(cols)
        return {name: E.DeviceTable(name, next(iter(c.values())).shape[0], {k: t.data_ptr() for k, t in c.items()})
                for name, c in cols.items()}

    def __del__(self):
        for f in self.close:
            try:
                f()
            except Exception:
                pass


def prepare(case, seed):
    ctx = _ctx()
    st = State(case)
    st.ctx = ctx
    kind = case["kind"]
    if kind == "scan":
        st.dev = st.tables(_fact(case["rows"], seed))
    elif kind == "join":
        st.dev = st.tables(_join_tables(case["a"], case["b"], seed))
    elif kind == "group":
        st.dev = st.tables(_group_table(case["rows"], case["skew"], case["groups"], case["cut"], seed))
        if case["sizing"] == "learned":
            st.est = EST.CardinalityEstimator(ctx).load()
    elif kind == "like":
        cols, st.w1, st.w2 = _text_tables(case["rows"], case["a"], seed)
        st.dev = st.tables(cols)
    elif kind == "anti":
        a, b = _dims(_gen(seed), case["a"], case["b"])
        st.dev = st.tables({"A": a, "B": b})
    elif kind == "batch":
        w = B.Workload3(ctx, B.workload3(case["pipes"], case["scale"], seed=int(seed) % 1_000_000), lds_cap=4096)
        for s in w.specs:                      # body settings the batch command documents (--set 4,12,2)
            w.batch_launch[s.index] = (256, 4, 12) if s.kind == "agg" else (256, 2, 10)
        st.w, st.b = w, w.build_batch(1024, 131_072, fold_rows=32_768)
        st.b.capture()
        st.close = [st.b.close, w.close]
        st.out = np.zeros((5, len(w.specs) * 4097), np.int64)
        st.used = 0
    else:
        st.db = T.TpchDB(ctx, _tpch_host(case["sf"], int(seed) % 1_000_000))
        for t in ("lineitem", "orders", "customer"):
            st.db.device(t)
        st.close = [st.db.free]
    n = len(case["queries"].split()) if kind in ("tpch", "sql") else 1
    st.ex = [E.HipGenericExecutor(ctx) for _ in range(n)]
    torch.cuda.synchronize()
    return st


def _padded(a, n):
    """`a` followed by zeros to a length that is the same for inputs of every seed."""
    return a if len(a) >= n else np.concatenate([a, np.zeros((n - len(a),) + a.shape[1:], a.dtype)])


def _csv(text, n):
    return np.frombuffer(text.encode().ljust(n, b"\0"), np.uint8)


#: Result rows of a kind that has few: buckets, the top 10, bins of the histogram, segments.
ROWS = {"scan": 6, "join": 10, "like": 64, "anti": 5}


def _arrays(columns, canonical, rows):
    """A result's columns as arrays of whole numbers (128-bit ones as low and high words; text is in the canonical CSV)."""
    out = {}
    for k, v in columns.items():
        if v.dtype != object:
            out[k] = _padded(v, rows)
        elif not isinstance(v[0], str):
            out[k] = _padded(np.array([(int(x) & 0xFFFFFFFF, int(x) >> 32) for x in v], dtype=np.int64), rows)
    out["csv"] = _csv(canonical, 256 + 256 * rows if rows <= 64 else 64 + 72 * rows if canonical else 0)
    return out


def run(st):
    c, ctx = st.case, st.ctx
    kind = c["kind"]
    if kind == "scan":
        r = Q.run_q1(ctx, st.dev, c["cutoff"], executor=st.ex[0]).result
    elif kind == "join":
        r = Q.run_q3(ctx, st.dev, c["seg"], c["date"], executor=st.ex[0]).result
    elif kind == "group":
        cut = c["cut"] or None
        if c["sizing"] == "learned":
            r = EST.run_groupby_learned(ctx, st.dev, st.est, 1, 3 * c["groups"], val_cut=cut, executor=st.ex[0])[0].result
        else:
            r = Q.run_groupby(ctx, st.dev, prepass=True, variant=c["variant"], key_min=1, key_max=3 * c["groups"],
                              val_cut=cut, lds_slots=4096 if c["variant"] == "part" else 2048, executor=st.ex[0]).result
    elif kind == "like":
        r = Q.run_q13(ctx, st.dev, st.w1, st.w2, negate=c["negate"], executor=st.ex[0]).result
    elif kind == "anti":
        r = Q.run_q22(ctx, st.dev, c["lo"], c["hi"], executor=st.ex[0]).result
    elif kind == "batch":
        st.b.run(graph=True)
        i = 0
        for s, p in zip(st.w.specs, st.w.results()):      # a pipeline's rows: their number, then its columns
            cols = ("key", "count", "sum", "min", "max") if s.kind == "agg" else ("rows", "sum_val")
            n = len(p[cols[0]])
            st.out[0, i] = n
            i += 1
            for j, k in enumerate(cols):
                st.out[j, i:i + n] = p[k]
            i += n
        st.out[:, i:st.used] = 0
        st.used = i
        return st.out
    else:
        qs = c["queries"].split()
        if kind == "tpch":
            runs = [T.run(ctx, st.db, q, executor=ex) for q, ex in zip(qs, st.ex)]
        else:
            runs = [S.run_sql(ctx, st.db, SQL[q], executor=ex) for q, ex in zip(qs, st.ex)]
        return {q: _csv(x.canonical, 2048) for q, x in zip(qs, runs)}
    return _arrays(r.columns, r.canonical, ROWS.get(kind) or c["groups"])


def work(case):
    """Every column the query reads once, every result row written once; operations are not what bounds any of these."""
    kind = case["kind"]
    if kind == "scan":
        return {"bytes": 26 * case["rows"], "flops": 12 * case["rows"]}
    if kind == "join":
        f = 4 * case["b"]
        return {"bytes": 5 * case["a"] + 12 * case["b"] + 20 * f, "flops": 3 * f}
    if kind == "group":
        return {"bytes": 12 * case["rows"] + 40 * case["groups"], "flops": 4 * case["rows"]}
    if kind == "like":
        return {"bytes": 29 * case["rows"] + 4 * case["a"], "flops": W.S_WIDTH * case["rows"]}
    if kind == "anti":
        return {"bytes": 8 * case["b"] + 5 * case["a"], "flops": 2 * case["b"]}
    if kind == "batch":
        rows = case["pipes"] * case["scale"] * (1e7 - 1e4) / (3 * math.log(10))
        return {"bytes": rows * (17 + 12) / 2, "flops": 4 * rows}
    lines, orders, cust = 6_000_000 * case["sf"], 1_500_000 * case["sf"], 150_000 * case["sf"]
    per = {"Q1": 38 * lines, "Q4": 12 * lines + 9 * orders, "Q6": 28 * lines, "Q13": 83 * orders + 4 * cust,
           "Q22": 27 * cust + 4 * orders, "Q12": 18 * lines + 5 * orders}
    return {"bytes": sum(per[q] for q in case["queries"].split()), "flops": 4 * lines}


def tolerance(case):
    return "exact"      # whole numbers and bytes throughout


def _np(t):
    return t.cpu().numpy()


def _by_key(key, val, keys):
    """key, count, sum, min, max of every key present, ascending."""
    key = key.to(torch.int64)
    cnt = torch.zeros(keys + 1, dtype=torch.int64, device="cuda").index_add_(0, key, torch.ones_like(key))
    tot = torch.zeros_like(cnt).index_add_(0, key, val)
    mn = torch.full_like(cnt, 2**62).scatter_reduce_(0, key, val, "amin")
    mx = torch.full_like(cnt, -2**62).scatter_reduce_(0, key, val, "amax")
    at = cnt.nonzero().reshape(-1)
    return {"key": _np(at), "count": _np(cnt[at]), "sum": _np(tot[at]), "min": _np(mn[at]), "max": _np(mx[at]), "csv": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "scan":
        f = _fact(case["rows"], seed)["F"]
        keep = f["f_date"] <= case["cutoff"]
        p, d, t = (f[k][keep].to(torch.int64) for k in ("f_price", "f_disc", "f_tax"))
        q = f["f_qty"][keep].to(torch.int64)
        fl, stt = f["f_flag"][keep], f["f_status"][keep]
        bucket = torch.where(fl == 65, 0, torch.where(fl == 78, 2, 4)) + (stt != 70).to(torch.int64)
        charge = p * (100 - d) * (100 + t)
        out = {k: [] for k in ("sum_qty", "sum_base_price", "sum_disc_price", "sum_charge", "sum_disc", "count_order",
                               "avg_qty", "avg_price", "avg_disc")}
        pair = lambda v: (v & 0xFFFFFFFF, v >> 32)  # noqa: E731
        for b in range(6):
            m = bucket == b
            n = int(m.sum())
            if not n:
                continue
            sq, sp, sd = int(q[m].sum()), int(p[m].sum()), int(d[m].sum())
            out["sum_qty"].append(sq)
            out["sum_base_price"].append(sp)
            out["sum_disc_price"].append(int((p[m] * (100 - d[m])).sum()))
            out["sum_charge"].append(pair((int((charge[m] >> 24).sum()) << 24) + int((charge[m] & 0xFFFFFF).sum())))
            out["sum_disc"].append(sd)
            out["count_order"].append(n)
            for k, v in (("avg_qty", sq), ("avg_price", sp), ("avg_disc", sd)):
                out[k].append(pair(v * 10**6 // n))
        return dict({k: _padded(np.array(v, dtype=np.int64), 6) for k, v in out.items()}, csv=None)
    if kind == "join":
        tb = _join_tables(case["a"], case["b"], seed)
        a, b, f = tb["A"], tb["B"], tb["F"]
        seg = torch.zeros(case["a"] + 1, dtype=torch.bool, device="cuda")
        seg[a["a_key"].to(torch.int64)] = a["a_seg"] == case["seg"]
        date = torch.full((case["b"] + 1,), -1, dtype=torch.int64, device="cuda")
        ok = (b["b_date"] < case["date"]) & seg[b["b_fkey"].to(torch.int64)]
        date[b["b_key"][ok].to(torch.int64)] = b["b_date"][ok].to(torch.int64)
        fk = f["f_fkey"].to(torch.int64)
        m = (f["f_date"] > case["date"]) & (date[fk] >= 0)
        rev = torch.zeros(case["b"] + 1, dtype=torch.int64, device="cuda")
        rev.index_add_(0, fk[m], f["f_price"][m] * (100 - f["f_disc"][m].to(torch.int64)))
        top = torch.topk(rev, min(64, rev.numel())).indices
        rows = sorted((-int(rev[k]), int(date[k]), int(k)) for k in top if int(rev[k]) > 0)[:10]
        key, rev, day = ([r[2] for r in rows], [-r[0] for r in rows], [r[1] for r in rows])
        return {"b_key": _padded(np.array(key), 10), "revenue": _padded(np.array(rev), 10),
                "b_date": _padded(np.array(day), 10), "csv": None}
    if kind == "group":
        g = _group_table(case["rows"], case["skew"], case["groups"], case["cut"], seed)["G"]
        m = g["g_val"] < (case["cut"] or 1 << 62)
        return _by_key(g["g_key"][m], g["g_val"][m], 3 * case["groups"])
    if kind == "anti":
        a, b = _dims(_gen(seed), case["a"], case["b"])
        hit = torch.zeros(case["a"] + 1, dtype=torch.bool, device="cuda")
        hit[b["b_fkey"][(b["b_date"] >= case["lo"]) & (b["b_date"] < case["hi"])].to(torch.int64)] = True
        m = ~hit[a["a_key"].to(torch.int64)]
        k, s = a["a_key"][m].to(torch.int64), a["a_seg"][m].to(torch.int64)
        n, t = (torch.zeros(5, dtype=torch.int64, device="cuda").index_add_(0, s, v) for v in (torch.ones_like(k), k))
        at = n.nonzero().reshape(-1)
        return {"num_keys": _padded(_np(n[at]), 5), "sum_keys": _padded(_np(t[at]), 5), "csv": None}
    return None         # text matching and whole plans: plain torch says nothing of them in a few lines
