"""The wildcard/edge-label join where CSR rows are read four entries at a time: hubs of fewer, exactly
and more than four and eight neighbours on both sides, edges listed twice with another label (the
first counts), and molecules over 64 nodes, against the CPU oracle.  Whole numbers: equality."""
import numpy as np
import pytest

from oracle import oracle as O
from sigmo_amd import capi
from tests.test_gpu_wildcard import _gpu_wildcard

pytestmark = pytest.mark.gpu

LEAVES = [7, 8, 9, 10, 11]


def _star(rng, leaves, nodes, wild=False, twice=False):
    """A hub of `leaves` neighbours, the last of which goes on as a path up to `nodes` nodes."""
    lab = [6] + [LEAVES[i % 5] for i in range(nodes - 1)]
    if wild:
        lab[int(rng.integers(1, leaves + 1))] = 255
    edges = [(0, i) for i in range(1, leaves + 1)] + [(i, i + 1) for i in range(leaves, nodes - 1)]
    bonds = [int(b) for b in rng.choice([1, 1, 1, 2], len(edges))]
    if twice:
        edges.append(edges[leaves // 2])
        bonds.append(3 - bonds[leaves // 2])
    return lab, edges, bonds


@pytest.mark.parametrize("leaves", [1, 3, 4, 5, 7, 8, 9])
@pytest.mark.parametrize("nodes", [24, 66])
def test_rows_of_four(ctx, leaves, nodes):
    rng = np.random.default_rng(10 * leaves + nodes)
    qs = [_star(rng, leaves, leaves + 1 + extra, wild, twice) for extra in (0, 2) for wild in (False, True) for twice in (False, True)]
    ms = [_star(rng, max(leaves, d), nodes, False, twice) for d in (leaves, 4, 5, 8, 9) for twice in (False, True) for _ in range(3)]
    qh, dh = capi.HostGraphs.from_edge_lists(qs), capi.HostGraphs.from_edge_lists(ms)
    q, d = qh.arrays(), dh.arrays()
    for find_first in (True, False):
        words, off, idx, total, counts = _gpu_wildcard(ctx, qh, dh, 1, find_first)
        o_total, o_counts = O.join_wildcard(q, d, words, off, idx, find_first)
        np.testing.assert_array_equal(counts, o_counts, err_msg=f"find_first={find_first}")
        assert total == o_total
