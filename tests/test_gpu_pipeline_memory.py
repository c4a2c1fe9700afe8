"""The plain pipeline where the device has memory for its level planes or for its pair arrays, not for
both: it runs, as it does level by level.  Whole numbers: equality."""
import numpy as np
import pytest
import torch

from sigmo_amd import capi

pytestmark = pytest.mark.gpu


def test_planes_give_way_to_the_pairs(ctx):
    # 400,000 molecules, 16 query labels and R = 8: 64 bytes of planes per node, 614 MB; 40 query graphs:
    # 18 bytes per possible pair, 288 MB
    R = 8
    rng = np.random.default_rng(0)
    qh = capi.HostGraphs.from_edge_lists([([int(x) for x in rng.integers(0, 16, 3)], [(0, 1), (1, 2)]) for _ in range(38)]
                                         + [(list(range(16)), [(i, i + 1) for i in range(15)]), ([8, 8, 8], [(0, 1), (1, 2)])])
    qd, dd = capi.DeviceGraph(ctx, qh), capi.DeviceGraph(ctx, capi.HostGraphs.molecules(5, 400_000, capi.SIZE_NORMAL))
    free = capi.Pipeline(ctx, qd, dd)
    want = free.execute(R, True), free.pairs()
    assert want[0]["gmcr_pairs"] > 100_000
    free.free()
    p = capi.Pipeline(ctx, qd, dd)
    planes = 64 * dd.total_nodes
    torch.empty(1, device="cuda:0")
    ballast = []
    try:
        for _ in range(3):  # a large allocation leaves more than it was asked to
            left = torch.cuda.mem_get_info(0)[0] - planes - (140 << 20)
            if left > 0:
                ballast.append(torch.empty(left, dtype=torch.uint8, device="cuda:0"))
        for _ in range(2):
            r = p.execute(R, True)
            assert (r["num_matches"], r["gmcr_pairs"]) == (want[0]["num_matches"], want[0]["gmcr_pairs"])
            for a, b in zip(p.pairs(), want[1]):
                np.testing.assert_array_equal(a, b)
    finally:
        ballast.clear()
        torch.cuda.empty_cache()
    assert p.execute(R, True)["num_matches"] == want[0]["num_matches"]  # with the planes again
