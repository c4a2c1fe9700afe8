"""The lane join at the edges of its levels in LDS (queries of 8 and 12 nodes), of its position words
(molecules of 64 and 128 nodes) and of its two-pass form (2^24 pairs), against the CPU oracle and the
one-pass form.  All results are whole numbers: equality."""
import numpy as np
import pytest

from oracle import oracle as O
from sigmo_amd import capi

pytestmark = pytest.mark.gpu

R = 2


def _graph(rng, n, extra):
    """A connected graph of n nodes: a path with random chords, two labels."""
    edges = {(i, i + 1) for i in range(n - 1)}
    while len(edges) < n - 1 + extra:
        a, b = sorted(int(x) for x in rng.integers(0, n, 2))
        if a != b:
            edges.add((a, b))
    return [int(x) for x in rng.integers(6, 8, n)], sorted(edges)


def _path(n):
    return [6] * n, [(i, i + 1) for i in range(n - 1)]


def _queries(rng, ks):
    """Paths of one label (which match deep), and of two, without and with a chord."""
    out = []
    for k in ks:
        out.append(_path(k))
        out.append(_graph(rng, k, 0))
        if k > 3:
            out.append(_graph(rng, k, 1))
    return out


@pytest.mark.parametrize("ks", [(2, 3, 7, 8), (8, 9), (9, 11, 12, 13), (5, 20, 31, 32)])
@pytest.mark.parametrize("ns", [(2, 9, 31, 32, 33), (63, 64), (65, 90, 128), (20, 64, 65)])
def test_levels_and_words(ctx, ks, ns):
    rng = np.random.default_rng(sum(ks) * 1000 + sum(ns))
    qh = capi.HostGraphs.from_edge_lists(_queries(rng, ks))
    dh = capi.HostGraphs.from_edge_lists([g for n in ns for g in [_path(n)] + [_graph(rng, n, n // 8) for _ in range(12)]])
    qd, dd = capi.DeviceGraph(ctx, qh), capi.DeviceGraph(ctx, dh)
    ref = O.pipeline(qh.arrays(), dh.arrays(), R, modes=[True, False])
    db = capi.Database(ctx, dd, R)
    steps = {}
    for form in (capi.Pipeline(ctx, qd, dd), capi.Batch(ctx, db)):
        for mode, key in ((True, "first"), (False, "all")):
            r = form.execute(R, mode) if isinstance(form, capi.Pipeline) else form.run(qd, mode)
            off, idx, cnt = form.pairs()
            np.testing.assert_array_equal(off, ref["offsets"])
            np.testing.assert_array_equal(idx, ref["indices"])
            np.testing.assert_array_equal(cnt, ref[f"counts_{key}"])
            assert r["num_matches"] == ref[f"total_{key}"]
            assert steps.setdefault(key, r["dfs_steps"]) == r["dfs_steps"]


def test_two_passes_equal_one(ctx):
    # 4096 x 4100 pairs: the first run joins the pairs found (one pass), the second is sized for
    # every pair (two passes); molecules of at most 64 nodes keep the one-synchronisation path
    qh = capi.HostGraphs.queries(5, 4096, 4, 20, capi.SIZE_NORMAL, perturb_frac=0.2)
    dh = capi.HostGraphs.molecules(6, 4100, capi.SIZE_NORMAL)
    qd, dd = capi.DeviceGraph(ctx, qh), capi.DeviceGraph(ctx, dh)
    db = capi.Database(ctx, dd, 6)
    batch = capi.Batch(ctx, db)
    one = batch.run(qd, True)
    off, idx, cnt = batch.pairs()
    two = batch.run(qd, True)
    off2, idx2, cnt2 = batch.pairs()
    assert not one["one_sync"] and two["one_sync"] and one["gmcr_pairs"] < 1 << 24 <= qh.num_graphs * dh.num_graphs
    np.testing.assert_array_equal(off, off2)
    np.testing.assert_array_equal(idx, idx2)
    np.testing.assert_array_equal(cnt, cnt2)
    for k in ("num_matches", "matched_pairs", "gmcr_pairs", "dfs_steps"):
        assert one[k] == two[k], k
