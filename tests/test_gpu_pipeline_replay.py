"""A captured pipeline whose buffers a later execute outgrows: the level planes grow with the level count
(the graph keeps its own), the result arrays with the pairs found (the replay is refused).  Whole
numbers: equality."""
import numpy as np
import pytest

from sigmo_amd import capi

pytestmark = pytest.mark.gpu


def _same(a, b):
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("captured,executed", [(1, 6), (2, 8), (6, 2), (6, 9), (9, 6)])
def test_replay_after_an_execute_of_other_levels(ctx, captured, executed):
    qd = capi.DeviceGraph(ctx, capi.HostGraphs.queries(31, 40, 4, 12, capi.SIZE_NORMAL))
    dd = capi.DeviceGraph(ctx, capi.HostGraphs.molecules(31, 3001, capi.SIZE_NORMAL))
    p, fresh = capi.Pipeline(ctx, qd, dd), capi.Pipeline(ctx, qd, dd)
    want = {}
    for R in (captured, executed):
        r = fresh.execute(R, True)
        want[R] = r["num_matches"], r["gmcr_pairs"], fresh.pairs()
    p.capture(captured, True)
    for R in (executed, executed, 8):  # further growths, and none
        p.execute(R, True)
        if R == executed:
            _same(p.pairs(), want[R][2])
        for _ in range(2):
            r = p.replay()
            assert (r["num_matches"], r["gmcr_pairs"]) == want[captured][:2]
            _same(p.pairs(), want[captured][2])
    p.capture(executed, True)
    assert p.replay()["num_matches"] == want[executed][0]
    _same(p.pairs(), want[executed][2])


def test_replay_is_refused_once_its_arrays_are_gone(ctx):
    # molecules of more than 64 nodes: arrays sized by the pairs found
    qd = capi.DeviceGraph(ctx, capi.HostGraphs.queries(32, 60, 4, 16, capi.SIZE_LOGNORMAL))
    dd = capi.DeviceGraph(ctx, capi.HostGraphs.molecules(32, 2000, capi.SIZE_LOGNORMAL))
    p = capi.Pipeline(ctx, qd, dd)
    p.capture(6, True)
    first = p.replay()
    pairs = p.pairs()
    more = p.execute(0, True)
    assert more["gmcr_pairs"] > 1.5 * first["gmcr_pairs"]
    for _ in range(2):
        with pytest.raises(capi.SigmoError, match="capture"):
            p.replay()
    p.capture(6, True)
    assert p.replay()["num_matches"] == first["num_matches"]
    _same(p.pairs(), pairs)
