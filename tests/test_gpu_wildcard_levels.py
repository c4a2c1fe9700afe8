"""The wildcard/edge-label join at the edges of its levels in LDS (order positions 7 and 8), with the
node of most candidates first, in the middle and last, repeated CSR entries and molecules over 64
nodes, against the CPU oracle.  All results are whole numbers: equality."""
import numpy as np
import pytest

from oracle import oracle as O
from sigmo_amd import capi
from tests.test_gpu_wildcard import _gpu_wildcard

pytestmark = pytest.mark.gpu


def _path(labels, bonds):
    return labels, [(i, i + 1) for i in range(len(labels) - 1)], bonds


@pytest.mark.parametrize("k", [2, 7, 8, 9, 12, 20])
@pytest.mark.parametrize("n", [24, 64, 65, 128])
def test_levels_and_order(ctx, k, n):
    rng = np.random.default_rng(100 * k + n)
    # labels repeat every five nodes, so searches stay short; a wildcard node has most candidates: it
    # leads the matching order wherever it stands
    cycle = [6, 7, 8, 9, 10]
    qs = [_path([255 if i == at else cycle[i % 5] for i in range(k)], [1] * (k - 1)) for at in sorted({0, k // 2, k - 1})]
    qs.append(_path([cycle[i % 5] for i in range(k)], [1] * (k - 2) + [2]))
    ms = []
    for _ in range(6):
        lab, edges, bonds = _path([cycle[i % 5] for i in range(n)], [int(b) for b in rng.choice([1] * 9 + [2], n - 1)])
        for _ in range(n // 24):  # chords
            a, b = sorted(int(x) for x in rng.integers(0, n, 2))
            if a != b and (a, b) not in edges:
                edges.append((a, b))
                bonds.append(int(rng.integers(1, 3)))
        if n == 24:  # a bond listed twice, with another label the second time: the first counts
            edges.append(edges[3])
            bonds.append(3 - bonds[3])
        ms.append((lab, edges, bonds))
    qh, dh = capi.HostGraphs.from_edge_lists(qs), capi.HostGraphs.from_edge_lists(ms)
    q, d = qh.arrays(), dh.arrays()
    for find_first in (True, False):
        words, off, idx, total, counts = _gpu_wildcard(ctx, qh, dh, 1, find_first)
        o_total, o_counts = O.join_wildcard(q, d, words, off, idx, find_first)
        np.testing.assert_array_equal(counts, o_counts, err_msg=f"find_first={find_first}")
        assert total == o_total
