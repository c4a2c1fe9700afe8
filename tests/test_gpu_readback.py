"""Results read back through the context's pinned halves (2 MB each): sizes around one and two halves,
and three arrays that share a half.  Every pair of these wildcard searches survives, so the lists are
known: equality."""
import threading

import numpy as np
import pytest

from sigmo_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("molecules", [1, 8191, 8192, 8193, 16384, 20001])
def test_pairs_around_the_halves(ctx, molecules):
    # 64 two-node wildcard query graphs: 8,192 molecules give 2 MB of indices
    qh = capi.HostGraphs.from_edge_lists([([255, 255], [(0, 1)])] * 64)
    dh = capi.HostGraphs.from_edge_lists([([6, 7, 8][: 2 + i % 2], [(0, 1), (1, 2)][: 1 + i % 2]) for i in range(molecules)])
    qd, dd = capi.DeviceGraph(ctx, qh), capi.DeviceGraph(ctx, dh)
    forms = [capi.Batch(ctx, capi.Database(ctx, dd, 1)), capi.Pipeline(ctx, qd, dd)]
    forms[0].run(qd, True)
    forms[1].execute(1, True)
    got = {}

    def read(i):
        got[i] = forms[i % 2].pairs()

    threads = [threading.Thread(target=read, args=(i,)) for i in range(4)]  # calls of several threads take turns
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(4):
        off, idx, cnt = got[i]
        np.testing.assert_array_equal(off, np.arange(molecules + 1) * 64)
        np.testing.assert_array_equal(idx, np.tile(np.arange(64), molecules))
        np.testing.assert_array_equal(cnt, np.ones(64 * molecules))
