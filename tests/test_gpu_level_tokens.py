"""The plain pipeline where a query node has as many signature requirements as it can have (31: a
32-node query whose other nodes all differ in distance or label) besides a label that the sweep holds
no plane of, against the CPU oracle.  The molecule lacks the last requirement alone.  Whole numbers:
equality."""
import numpy as np
import pytest

from oracle import oracle as O
from sigmo_amd import capi

pytestmark = pytest.mark.gpu


def _two_rings(centre, leaves):
    """A centre, 16 neighbours labelled 0..15 and grandchildren labelled 0..leaves-1."""
    return [centre] + list(range(16)) + list(range(leaves)), [(0, i) for i in range(1, 17)] + [(1 + i, 17 + i) for i in range(leaves)]


def _beside(a, b):
    n = len(a[0])
    return a[0] + b[0], a[1] + [(u + n, v + n) for u, v in b[1]]


@pytest.mark.parametrize("centre", [20, 200, 255])
@pytest.mark.parametrize("R", [2, 6, 8])
def test_all_requirements_of_a_far_label(ctx, centre, R):
    query = _two_rings(centre, 15)
    assert len(query[0]) == 32
    # the second component has candidates for every node but the centre, whose label differs
    lacking = _beside(_two_rings(20, 14), _two_rings(21, 15))
    holding = _beside(_two_rings(20, 15), _two_rings(200, 15))
    qh = capi.HostGraphs.from_edge_lists([query, ([8, 7], [(0, 1)])])
    dh = capi.HostGraphs.from_edge_lists([lacking, holding, _two_rings(centre % 255, 15), _two_rings(centre % 255, 14)])
    qd, dd = capi.DeviceGraph(ctx, qh), capi.DeviceGraph(ctx, dh)
    ref = O.pipeline(qh.arrays(), dh.arrays(), R, modes=[True, False])
    for form in (capi.Pipeline(ctx, qd, dd), capi.Batch(ctx, capi.Database(ctx, dd, R))):
        for mode, key in ((True, "first"), (False, "all")):
            r = form.execute(R, mode) if isinstance(form, capi.Pipeline) else form.run(qd, mode)
            off, idx, cnt = form.pairs()
            np.testing.assert_array_equal(off, ref["offsets"])
            np.testing.assert_array_equal(idx, ref["indices"])
            np.testing.assert_array_equal(cnt, ref[f"counts_{key}"])
            assert r["num_matches"] == ref[f"total_{key}"]
