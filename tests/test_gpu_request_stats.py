"""Per-request statistics of a batch against the sums of its pairs: numbers of requests on both sides
of each change in the kernel's copies of the sums, empty requests among them, pair counts that are
no multiple of the four a thread takes, and more pairs than one turn of the grid."""
from __future__ import annotations

import numpy as np
import pytest

from sigmo_amd import capi
from tests._util import request_stats

pytestmark = pytest.mark.gpu


def _check(ctx, molecules, queries, kmax, splits):
    dd = capi.DeviceGraph(ctx, capi.HostGraphs.molecules(11, molecules, capi.SIZE_NORMAL))
    db = capi.Database(ctx, dd, 2)
    batch = capi.Batch(ctx, db)
    qd = capi.DeviceGraph(ctx, capi.HostGraphs.queries(11, queries, 4, kmax, capi.SIZE_NORMAL))
    r = batch.run(qd, find_first=False)
    off, idx, cnt = batch.pairs()
    for rgo in splits:
        got = batch.request_stats(rgo)
        assert [(p["matched_pairs"], p["embeddings"], p["hash"]) for p in got] == request_stats(off, idx, cnt, rgo), len(rgo) - 1
    return r["gmcr_pairs"]


def _split(rng, queries, n):
    """n requests over the query graphs, cut anywhere (the first, the last and others may be empty)."""
    return np.concatenate([[0], np.sort(rng.randint(0, queries + 1, n - 1)), [queries]]).astype(np.uint32)


def test_request_counts(ctx):
    rng = np.random.RandomState(0)
    splits = [_split(rng, 301, n) for n in (1, 2, 5, 6, 16, 17, 32, 33, 64, 65, 128, 129, 255, 256)]
    splits.append(np.array([0, 0, 301, 301], np.uint32))
    _check(ctx, 997, 301, 12, splits)


@pytest.mark.parametrize("molecules", [1, 2, 3, 7])
def test_few_pairs(ctx, molecules):
    _check(ctx, molecules, 5, 5, [[0, 5], [0, 2, 2, 5]])


def test_many_pairs(ctx):
    pairs = _check(ctx, 40_003, 250, 6, [[0, 250], [0, 1, 249, 250]])
    assert pairs > 2 * 256 * 4096  # more than one turn of two blocks per CU, four pairs a thread
