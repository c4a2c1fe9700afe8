"""The batched form's candidate arena: its demand follows the pairs that survive, not those that pass the
pre-test, in groups of which none, some and most survive, against the CPU oracle.  Whole numbers:
equality; the demand is bounded by the first sizing or the survivors' words."""
import numpy as np
import pytest

from oracle import oracle as O
from sigmo_amd import capi

pytestmark = pytest.mark.gpu

R = 2
PARTS = ([(0, 1), (0, 2), (0, 3)], [(0, 1), (0, 2), (1, 3), (1, 4), (2, 5)])  # a star; a path with side nodes
SPIDER = [(0, 1), (0, 2), (0, 3), (1, 4), (2, 5), (3, 6)]


def _graph(pieces, n):
    """Components of one label, filled up to n nodes with single ones."""
    edges, at = [], 0
    for e in pieces:
        edges += [(a + at, b + at) for a, b in e]
        at += 1 + max(max(x) for x in e)
    assert at <= n
    return [8] * n, edges


def _spider(rng, centre, extra):
    """The spider, or with its centre as node `centre` and `extra` nodes in a row at a leg."""
    if not extra:
        return [8] * 7, SPIDER
    edges = SPIDER + [(6 + i, 7 + i) for i in range(extra)]
    n = 7 + extra
    order = [x for x in rng.permutation(n) if x != 0]
    order.insert(min(centre, n - 1), 0)
    place = {int(x): i for i, x in enumerate(order)}
    return [8] * n, [(place[a], place[b]) for a, b in edges]


@pytest.mark.parametrize("n", [17, 40, 70])
@pytest.mark.parametrize("every", [0, 67, 5, 2])
def test_demand_follows_the_survivors(ctx, n, every):
    # The star has the largest count at distance 1, the path with side nodes the largest at distance 2;
    # the spider's centre needs both.  Every `every`-th molecule has a spider.
    rng = np.random.default_rng(n + every)
    ms = [_graph([*PARTS, SPIDER] if every and i % every == 0 else PARTS, n) for i in range({17: 12000, 40: 5000, 70: 3000}[n])]
    qs = [_spider(rng, i % 32, (25, 22, 0, 1)[i % 4]) for i in range(130)]
    qh, dh = capi.HostGraphs.from_edge_lists(qs), capi.HostGraphs.from_edge_lists(ms)
    qd, dd = capi.DeviceGraph(ctx, qh), capi.DeviceGraph(ctx, dh)
    ref = O.pipeline(qh.arrays(), dh.arrays(), R, modes=[True])
    assert (ref["total_first"] > 0) == (every > 0)
    batch = capi.Batch(ctx, capi.Database(ctx, dd, R))
    batch.tuning = {"filter_blocks_per_cu": 1}
    for sized in (False, True):  # the first run sizes the arena, and may be repeated for it
        ctx.reset_phases()
        r = batch.run(qd, True)
        off, idx, cnt = batch.pairs()
        np.testing.assert_array_equal(off, ref["offsets"])
        np.testing.assert_array_equal(idx, ref["indices"])
        np.testing.assert_array_equal(cnt, ref["counts_first"])
        assert r["filter_scans"] > 0.5 * len(qs) * len(ms)
        if not sized:
            continue
        assert r["arena_repeats"] == 0
        # the pair filter's bytes: inputs read once, survival bits and the arena's words written
        reads = (1 + 8 * R) * dd.total_nodes + qd.total_nodes * (1 + 2 * 16 * R) + len(qs) * (4 + 8 * R)
        words = (ctx.kernel_stats()["pair_filter"][2] - reads) / 8 - len(ms) * ((len(qs) + 63) // 64)
        k = np.array([len(lab) for lab, _ in qs])[idx]
        own = {17: (k + 3) // 4 * 2, 40: (k + 3) // 4 * 4, 70: (k + 1) // 2 * 4}[n].sum()
        # a run that overflows the first sizing keeps the survivors' words, half of each chunk at least
        slack = 2 * 2048 * 8 * 256  # 256 CUs x 8 wavefronts, two chunks each
        first = max(len(qs) * len(ms) // 8, 1 << 16) * (np.mean([len(lab) for lab, _ in qs]) + 1) * (2 if n > 64 else 1)
        assert words <= max(first, 2 * own) + slack, (words, own)


def test_first_sizing_near_the_largest_arena(ctx):
    # 2^29 pairs and one molecule of more than 64 nodes: the guess for 30-node queries is 4.16 G words of the
    # 2^32 that offsets reach, and the wavefronts' chunks come on top.  No pair passes the pre-test.
    rng = np.random.default_rng(0)
    path = [(i, i + 1) for i in range(29)]
    qh = capi.HostGraphs.from_edge_lists([([int(x) for x in rng.integers(0, 16, 30)], path) for _ in range(4100)])
    ones = 131_071
    dh = capi.HostGraphs.from_arrays(np.arange(ones + 1), np.zeros(ones + 1), np.zeros(0), rng.integers(0, 16, ones))
    dh = dh.concat(capi.HostGraphs.from_edge_lists([([8] * 65, path)]))
    dd = capi.DeviceGraph(ctx, dh)
    batch = capi.Batch(ctx, capi.Database(ctx, dd, 2))
    r = batch.run(capi.DeviceGraph(ctx, qh), True)
    assert r["gmcr_pairs"] == 0 and r["arena_repeats"] == 0
    few = batch.run(capi.DeviceGraph(ctx, capi.HostGraphs.from_edge_lists([([8, 8], [(0, 1)])])), True)
    assert few["gmcr_pairs"] == 1 and few["matched_pairs"] == 1
