"""bench.py's kernel statistics by launch: what one launch shared out equally is put together again."""
import bench

# what the library reports for one plain execute with R = 6: two launches, 1 + 6 and 1 + 5 equal shares
# (times are 32-bit before they are shared out)
SWEEP = {"sig_generate": (1, 2.0, 14.0), "sig_refine": (6, 12.0, 84.0), "filter": (1, 20.0, 30.0), "refine": (5, 100.0 + 5e-6, 150.0),
         "gmcr": (1, 50.0, 9.0), "join": (1, 60.0, 0.0), "pair_filter": (0, 0.0, 0.0)}


def test_shares_of_one_launch_are_one_kernel():
    got = bench.launched(SWEEP)
    assert got["filter_levels"] == (1, 120.0 + 5e-6, 180.0) and got["sig_levels"] == (1, 14.0, 98.0)
    assert not {"filter", "refine", "sig_generate", "sig_refine"} & set(got)
    assert max(got, key=lambda k: got[k][1]) == "filter_levels" and set(got) - {"join"} <= set(bench.HBM_KERNELS)
    assert bench.kernel_table(got, 1)["filter_levels"]["launches_per_step"] == 1.0
    assert abs(sum(v[1] for v in got.values()) - sum(v[1] for v in SWEEP.values())) < 1e-9


def test_kernels_of_their_own_stay():
    levels = {**SWEEP, "sig_refine": (9, 33.0, 84.0), "filter": (1, 20.0, 30.0), "refine": (8, 77.0, 150.0)}
    assert bench.launched(levels) == levels
    assert bench.launched({"join": (1, 1.0, 0.0)}) == {"join": (1, 1.0, 0.0)}

