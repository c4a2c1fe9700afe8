"""A join whose counts take more than one pinned half: the second copying thread does not occupy a core
while the join runs."""
import time

import numpy as np
import pytest

from sigmo_amd import capi

pytestmark = pytest.mark.gpu


def test_no_second_core_waits_for_the_join(ctx):
    # every pair of these wildcard searches survives: 2 M counts (8 MB), and the join takes about 90% of the call
    a = capi.HostGraphs.queries(2, 100, 10, 16, capi.SIZE_NORMAL).arrays()
    qh = capi.HostGraphs.from_arrays(a["graph_offsets"], a["row_offsets"], a["column_indices"], np.full_like(a["node_labels"], 255), a["edge_labels"])
    qd, dd = capi.DeviceGraph(ctx, qh), capi.DeviceGraph(ctx, capi.HostGraphs.molecules(1, 20_000, capi.SIZE_NORMAL))
    sig, cand = capi.Signature(ctx, dd.total_nodes, qd.total_nodes), capi.Candidates(ctx, qd.total_nodes, dd.total_nodes)
    capi.filter_candidates(ctx, qd, dd, sig, cand)
    gm = capi.GMCR(ctx)
    gm.generate(qd, dd, cand)
    assert gm.total == 2_000_000
    alone, _ = capi.join_candidates(ctx, qd, dd, cand, gm, True, per_pair=False)
    shares = []
    for _ in range(5):
        cpu, wall = time.process_time(), time.perf_counter()
        total, counts = capi.join_candidates(ctx, qd, dd, cand, gm, True)
        shares.append((time.process_time() - cpu) / (time.perf_counter() - wall))
        assert total == alone == int(counts.sum())
    assert min(shares) < 1.5, shares  # this thread waits for the stream; one more beside it made 1.97
