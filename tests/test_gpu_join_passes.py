"""The lane join on both sides of the pair count from which it takes two passes: a batch over it against
its halves, which are under it, pair by pair (whole numbers: equality)."""
from __future__ import annotations

import numpy as np
import pytest

from sigmo_amd import capi

pytestmark = pytest.mark.gpu

TWO_PASS_PAIRS = 3 << 21  # find-first; counting every embedding takes one pass on both sides here


@pytest.mark.parametrize("find_first", [True, False])
def test_two_passes_equal_one(ctx, find_first):
    queries, half = 801, 400
    qh = capi.HostGraphs.queries(21, queries, 4, 24, capi.SIZE_LOGNORMAL, ring_frac=0.2)
    dd = capi.DeviceGraph(ctx, capi.HostGraphs.molecules(21, 100_003, capi.SIZE_LOGNORMAL))
    batch = capi.Batch(ctx, capi.Database(ctx, dd, 6))

    def pairs(first, n):
        r = batch.run(capi.DeviceGraph(ctx, qh.slice(first, n)), find_first)
        off, idx, cnt = batch.pairs()
        mol = np.repeat(np.arange(len(off) - 1, dtype=np.int64), np.diff(off.astype(np.int64)))
        return r, mol * queries + idx.astype(np.int64) + first, cnt

    a, ka, ca = pairs(0, half)
    b, kb, cb = pairs(half, queries - half)
    assert max(ka.size, kb.size) < TWO_PASS_PAIRS
    whole, key, cnt = pairs(0, queries)
    assert key.size >= TWO_PASS_PAIRS
    ks = np.concatenate([ka, kb])
    order = np.argsort(ks, kind="stable")
    np.testing.assert_array_equal(key, ks[order])
    np.testing.assert_array_equal(cnt, np.concatenate([ca, cb])[order])
    for k in ("num_matches", "matched_pairs", "dfs_steps"):
        assert whole[k] == a[k] + b[k]
