"""The pipeline's one-sweep filter and both forms' requirement tests at their edges: counts around the
largest that LDS holds a plane of (4, and 8 for the most frequent label) and the saturated 15, more labels than LDS holds, strips of
2,048 data nodes, and level counts with and without the sweep; against the CPU oracle.  All results
are whole numbers: equality."""
import numpy as np
import pytest

from oracle import oracle as O
from sigmo_amd import capi

pytestmark = pytest.mark.gpu


def _star(leaves, centre=8, leaf=7, tail=0):
    """A star whose first leaf carries a path of `tail` more nodes."""
    edges = [(0, i) for i in range(1, leaves + 1)]
    labels = [centre] + [leaf] * leaves
    for t in range(tail):
        edges.append((1 if t == 0 else len(labels) - 1, len(labels)))
        labels.append(centre)
    return labels, edges


def _check(ctx, qs, ms, R, batched=True):
    qh, dh = capi.HostGraphs.from_edge_lists(qs), capi.HostGraphs.from_edge_lists(ms)
    qd, dd = capi.DeviceGraph(ctx, qh), capi.DeviceGraph(ctx, dh)
    ref = O.pipeline(qh.arrays(), dh.arrays(), R, modes=[True])
    forms = [capi.Pipeline(ctx, qd, dd)] + ([capi.Batch(ctx, capi.Database(ctx, dd, R))] if batched else [])
    for form in forms:
        for _ in range(2):
            r = form.execute(R, True) if isinstance(form, capi.Pipeline) else form.run(qd, True)
            off, idx, cnt = form.pairs()
            np.testing.assert_array_equal(off, ref["offsets"])
            np.testing.assert_array_equal(idx, ref["indices"])
            np.testing.assert_array_equal(cnt, ref["counts_first"])
            assert r["num_matches"] == ref["total_first"]


@pytest.mark.parametrize("R", [1, 2, 3])
def test_counts_around_the_near_planes_and_saturation(ctx, R):
    counts = (1, 2, 3, 4, 5, 6, 8, 9, 14, 15, 16, 20, 30)
    qs = [_star(c) for c in counts if c < 32] + [_star(c, tail=2) for c in counts if c < 29]
    ms = [_star(c, tail=t) for c in counts for t in (0, 1, 3)] + [_star(c, tail=40) for c in (3, 5, 16, 60)]
    qs += [_star(c, leaf=6) for c in (4, 5, 8, 9)]  # a label with planes up to 4 only
    ms += [_star(c, leaf=6) for c in (4, 5, 7, 8, 9, 20)]
    _check(ctx, qs, ms, R)


@pytest.mark.parametrize("R,batched", [(1, True), (6, True), (8, True), (9, False), (12, False)])
def test_labels_strips_and_level_counts(ctx, R, batched):
    rng = np.random.default_rng(R)

    def tree(n, labels):
        return [int(labels[x]) for x in rng.integers(0, len(labels), n)], [(int(rng.integers(max(0, i - 3), i)), i) for i in range(1, n)]

    ms = [tree(int(n), list(range(2 + i % 15))) for i, n in enumerate(rng.choice([7, 24, 31, 32, 33, 64, 70], 170))]  # > 2 strips
    qs = [([a, b], [(0, 1)]) for a in (0, 5, 15) for b in range(16)] + [tree(k, [0, 1, 2, 3]) for k in (3, 4, 5, 8)]
    qs += [([255, 3], [(0, 1)]), ([200, 3], [(0, 1)])]
    _check(ctx, qs, ms, R, batched)


def test_query_labels_without_counts(ctx):
    # no query label below 16: nothing to refine
    ms = [([20, 21, 20], [(0, 1), (1, 2)]), ([20, 8, 21], [(0, 1), (1, 2)])] * 40
    _check(ctx, [([20, 21], [(0, 1)]), ([255, 255, 255], [(0, 1), (1, 2)])], ms, 3)
