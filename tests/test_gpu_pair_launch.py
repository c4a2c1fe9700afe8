"""The pair evaluation's launch on both sides of its choices, against the CPU oracle: one to eight blocks to
a group's query graphs (few groups, 8 to 40 query graphs), items that are all shared out beforehand
or claimed from the cursor (more groups than blocks), and both scatters (64 and 65 query graphs).
Whole numbers: equality."""
import numpy as np
import pytest

from oracle import oracle as O
from sigmo_amd import capi

pytestmark = pytest.mark.gpu


def _trees(rng, count, lo, hi):
    out = []
    for n in rng.integers(lo, hi + 1, count):
        out.append(([int(x) for x in rng.choice([8, 8, 7, 6], n)], [(int(rng.integers(max(0, i - 3), i)), i) for i in range(1, n)]))
    return out


# groups of 64 molecules x parts: 2 x 1, 2 x 2, 2 x 4, 2 x 8 (fewer items than blocks), 300 x 1 (256 blocks:
# 44 claimed), 150 x 4 (600 items, 344 claimed), 1,100 x 1 (768 shared out, 332 claimed)
@pytest.mark.parametrize("molecules,queries,blocks", [(100, 8, 0), (100, 9, 0), (100, 17, 0), (100, 40, 0), (100, 64, 0), (100, 65, 0),
                                                      (19_200, 5, 1), (9_600, 33, 1), (70_400, 3, 1), (70_400, 3, 0)])
def test_shares_and_claims(ctx, molecules, queries, blocks):
    rng = np.random.default_rng(molecules + queries)
    qh = capi.HostGraphs.from_edge_lists(_trees(rng, queries, 2, 5))
    dh = capi.HostGraphs.from_edge_lists(_trees(rng, molecules, 2, 9))
    qd, dd = capi.DeviceGraph(ctx, qh), capi.DeviceGraph(ctx, dh)
    ref = O.pipeline(qh.arrays(), dh.arrays(), 3, modes=[True])
    batch = capi.Batch(ctx, capi.Database(ctx, dd, 3))
    batch.tuning = {"filter_blocks_per_cu": blocks, "filter_claim": 5, "filter_mode": 2}  # the last two are accepted and ignored
    for _ in range(2):
        r = batch.run(qd, True)
        off, idx, cnt = batch.pairs()
        np.testing.assert_array_equal(off, ref["offsets"])
        np.testing.assert_array_equal(idx, ref["indices"])
        np.testing.assert_array_equal(cnt, ref["counts_first"])
        assert r["num_matches"] == ref["total_first"] > 0
