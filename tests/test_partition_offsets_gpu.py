"""The partitioned group-by's offsets pass at count partitions per table
partition of 1, a few, 64 and beyond, table partitions fewer and more than a
block's lanes, and block sizes below the planned one: against a sort."""

import numpy as np
import pytest

from gpudbmetalcodegen_amd import queries as Q
from helpers import group_rows

pytestmark = pytest.mark.gpu


# key range (count partitions) against distinct keys (table partitions)
@pytest.mark.parametrize("groups,span,block", [(10, 100, 1024), (1000, 4_000_000, 1024), (9000, 4_000_000, 256),
                                               (60_000, 500_000, 64), (60_000, 4_000_000, 1024), (300_000, 300_000, 512),
                                               (300_000, 3_000_000, 1024)])
def test_offsets(ctx, groups, span, block):
    print(groups, span, block, flush=True)
    r = np.random.default_rng(groups + span)
    ids = np.sort(r.choice(span, groups, replace=False)) + 1
    keys = np.concatenate([ids, r.choice(ids, 3 * groups)]).astype(np.int32)
    G = {"g_key": r.permutation(keys), "g_val": r.integers(-5000, 5000, keys.size)}
    dev = Q.upload_tables(ctx, {"G": G})
    try:
        run = Q.run_groupby(ctx, dev, prepass=True, variant="part", lds_slots=1024, key_min=1, key_max=span)
        run.plan.set_launch("GBP_offsets", block, 1)
        run = Q.run_groupby(ctx, dev, prepass=True, variant="part", lds_slots=1024, key_min=1, key_max=span)
        run.plan.set_launch("GBP_offsets", 1024, 1)
        for c, e in group_rows(G).items():
            assert np.array_equal(run.result.columns[c], e), c
    finally:
        dev["G"].free(ctx)
