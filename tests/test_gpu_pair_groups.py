"""The batched form's pair evaluation at the edges of its 64-lane groups (64, 32 or 16 molecules by size
class, the last of a class short), of the labels whose planes LDS holds, and of its 64-query words,
against the CPU oracle.  All results are whole numbers: equality."""
import numpy as np
import pytest

from oracle import oracle as O
from sigmo_amd import capi

pytestmark = pytest.mark.gpu


def _graph(rng, n, labels, chords=0):
    """A random tree of n nodes (degree <= 4) with a few chords."""
    edges, deg = set(), [0] * n
    for i in range(1, n):
        j = int(rng.choice([x for x in range(max(0, i - 6), i) if deg[x] < 4] or [i - 1]))
        edges.add((j, i))
        deg[i] += 1
        deg[j] += 1
    for _ in range(chords):
        a, b = sorted(int(x) for x in rng.integers(0, n, 2))
        if a != b:
            edges.add((a, b))
    return [int(labels[x]) for x in rng.integers(0, len(labels), n)], sorted(edges)


def _check(ctx, qs, ms, R):
    qh, dh = capi.HostGraphs.from_edge_lists(qs), capi.HostGraphs.from_edge_lists(ms)
    qd, dd = capi.DeviceGraph(ctx, qh), capi.DeviceGraph(ctx, dh)
    ref = O.pipeline(qh.arrays(), dh.arrays(), R, modes=[True, False])
    batch = capi.Batch(ctx, capi.Database(ctx, dd, R))
    for rep in range(2):  # the second run takes the path sized by the first
        for mode, key in ((True, "first"), (False, "all")):
            r = batch.run(qd, mode)
            off, idx, cnt = batch.pairs()
            np.testing.assert_array_equal(off, ref["offsets"])
            np.testing.assert_array_equal(idx, ref["indices"])
            np.testing.assert_array_equal(cnt, ref[f"counts_{key}"])
            assert r["num_matches"] == ref[f"total_{key}"] and r["filter_scans"] >= r["gmcr_pairs"]


@pytest.mark.parametrize("small,mid,wide", [(1, 0, 0), (63, 31, 15), (64, 32, 16), (65, 33, 17), (0, 1, 0), (0, 0, 1), (130, 0, 20)])
def test_group_sizes(ctx, small, mid, wide):
    rng = np.random.default_rng(small * 10000 + mid * 100 + wide)
    sizes = [int(x) for x in rng.integers(1, 33, small)] + [int(x) for x in rng.choice([33, 40, 63, 64], mid)] + \
        [int(x) for x in rng.choice([65, 96, 97, 128], wide)]
    ms = [_graph(rng, n, [8, 8, 7], n // 10) for n in rng.permutation(sizes)]
    qs = [_graph(rng, k, [8, 8, 7]) for k in (2, 3, 3, 4, 5, 6, 9)] + [([255, 8], [(0, 1)]), ([8, 255, 8], [(0, 1), (1, 2)])]
    _check(ctx, qs, ms, 4)


@pytest.mark.parametrize("count", [1, 63, 64, 65, 129])
def test_mask_blocks(ctx, count):
    # query sizes around the four masks of a 16-byte store, in all three mask widths
    rng = np.random.default_rng(count)
    ms = [_graph(rng, int(n), [8, 7, 6, 8], int(n) // 12) for n in rng.choice([9, 20, 32, 33, 50, 64, 65, 100, 128], 170)]
    qs = []
    for i in range(count):  # connected parts of the molecules: a node and those that follow it in its tree
        lab, edges = ms[int(rng.integers(0, len(ms)))]
        k = min(len(lab), 2 + i % 16)
        nodes = [int(rng.integers(0, len(lab)))]
        while len(nodes) < k:
            nodes += [b if a in nodes else a for a, b in edges if (a in nodes) != (b in nodes)][: k - len(nodes)]
            nodes = list(dict.fromkeys(nodes))
        qs.append(([lab[x] for x in nodes], [(nodes.index(a), nodes.index(b)) for a, b in edges if a in nodes and b in nodes]))
    _check(ctx, qs, ms, 3)


@pytest.mark.parametrize("R", [1, 6, 8])
def test_more_labels_than_lds_holds(ctx, R):
    rng = np.random.default_rng(R)
    labels = list(range(16))
    ms = [_graph(rng, int(n), labels[: 2 + i % 15], 1) for i, n in enumerate(rng.choice([12, 30, 50, 64, 70, 128], 150))]
    ms += [_graph(rng, 20, [3, 17, 200], 1) for _ in range(20)]  # labels without signature counts
    qs = []
    for _ in range(70):  # over one 64-query word: connected parts of the molecules, and single edges
        lab, edges = ms[int(rng.integers(0, len(ms)))]
        a, b = edges[int(rng.integers(0, len(edges)))]
        more = [e for e in edges if (a in e or b in e) and e != (a, b)][: int(rng.integers(0, 4))]
        nodes = sorted({x for e in [(a, b)] + more for x in e})
        qs.append(([lab[x] for x in nodes], [(nodes.index(x), nodes.index(y)) for x, y in [(a, b)] + more]))
    _check(ctx, qs, ms, R)
