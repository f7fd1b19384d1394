"""LIKE '%w1%w2%' by the words' first four bytes: small alphabets, so heads
match where words do not (the automata decide then), words of every length
class, words with a NUL in them (which match nothing, also where the bytes
after a value's end hold them), values ended by a NUL with bytes after it; and
counts whose histogram crosses the register bins. Against the oracle, both
signs."""

import numpy as np
import pytest

import oracle
from gpudbmetalcodegen_amd import queries as Q

pytestmark = pytest.mark.gpu

WORDS = [b"", b"a", b"ab", b"aba", b"abab", b"ababa", b"aaaab", b"abababab", b"baaaaaaab", b"ababababababababababab",
         b"a\0", b"a\0a", b"aaaaa\0a"]


@pytest.mark.parametrize("alphabet", [b"a", b"ab", b"abc"])
@pytest.mark.parametrize("n", [1, 4097])
def test_like_small_alphabets(ctx, alphabet, n):
    r = np.random.default_rng(n + len(alphabet))
    text = np.frombuffer(alphabet, np.uint8)[r.integers(0, len(alphabet), (n, 25))].copy()
    ends = r.integers(0, 40, n)
    for i in range(n):
        if ends[i] < 25:
            text[i, ends[i]] = 0                     # the bytes after it stay: not part of the value
            if r.random() < 0.5:
                text[i, ends[i]:] = 0
    n_a = 50
    S = {"s_fkey": r.integers(1, n_a + 1, n).astype(np.int32), "s_text": text}
    A = {"a_key": np.arange(1, n_a + 1, dtype=np.int32), "a_seg": np.zeros(n_a, np.uint8)}
    dev = Q.upload_tables(ctx, {"S": S, "A": A})
    ex = None
    try:
        for w1 in WORDS:
            for w2 in WORDS:
                for negate in (False, True):
                    run = Q.run_q13(ctx, dev, w1, w2, negate=negate, executor=ex)
                    ex = run.executor
                    exp = oracle.q13(S, A, n_a, w1, w2, negate=negate)
                    got = {k: [int(x) for x in v] for k, v in run.result.columns.items()}
                    assert got == {k: v.tolist() for k, v in exp.items()}, (w1, w2, negate)
    finally:
        for t in dev.values():
            t.free(ctx)


@pytest.mark.parametrize("n_a,n_b", [(31, 1000), (32, 1), (4095, 70_001), (100_003, 1_000_003)])
def test_anti_join_by_flags_equals_bitmap(ctx, n_a, n_b, monkeypatch):
    """Referenced keys as packed byte flags: key ranges around whole bitmap
    words, keys outside the range, and no referencing row at all."""
    r = np.random.default_rng(n_a)
    A = {"a_key": (r.permutation(n_a) + 1).astype(np.int32), "a_seg": r.integers(0, 5, n_a).astype(np.uint8)}
    B = {"b_key": np.arange(1, n_b + 1, dtype=np.int32), "b_fkey": r.integers(-3, n_a + 40, n_b).astype(np.int32),
         "b_date": r.integers(0, 2406, n_b).astype(np.int32)}
    dev = Q.upload_tables(ctx, {"A": A, "B": B})
    try:
        for lo, hi in [(0, 2406), (100, 300), (7, 7)]:
            monkeypatch.setattr(Q, "Q22_FLAG_ROWS", 1 << 40)
            plain = Q.run_q22(ctx, dev, lo, hi)
            monkeypatch.setattr(Q, "Q22_FLAG_ROWS", 0)
            flags = Q.run_q22(ctx, dev, lo, hi)
            assert "Q22_pack_bitmap" in flags.plan.phases() and "Q22_pack_bitmap" not in plain.plan.phases()
            assert flags.result.canonical == plain.result.canonical
            hit = np.isin(A["a_key"], B["b_fkey"][(B["b_date"] >= lo) & (B["b_date"] < hi)])
            assert int(np.sum(flags.result.columns["num_keys"])) == int((~hit).sum())
            assert int(np.sum(flags.result.columns["sum_keys"])) == int(A["a_key"][~hit].astype(np.int64).sum())
    finally:
        for t in dev.values():
            t.free(ctx)
