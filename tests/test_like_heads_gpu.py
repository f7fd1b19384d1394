"""LIKE '%w1%w2%' by the words' first four bytes: small alphabets, so heads
match where words do not (the automata decide then), words of every length
class, values ended by a NUL with bytes after it; and counts whose histogram
crosses the register bins. Against the oracle, both signs."""

import numpy as np
import pytest

import oracle
from gpudbmetalcodegen_amd import queries as Q

pytestmark = pytest.mark.gpu

WORDS = [b"", b"a", b"ab", b"aba", b"abab", b"ababa", b"aaaab", b"abababab", b"baaaaaaab", b"ababababababababababab"]


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
