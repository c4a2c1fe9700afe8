"""Timed workloads of the framework's public entry points.

Every case is one call sequence that a program makes in earnest: a screening run or a served
request of the batched form over a resident molecule database, the plain per-phase pipeline, the
per-phase calls themselves, or a pass over a molecule shard streamed from host memory.  Sizes and
distributions are those of the smoke test, the tests and bench.py's configurations (Normal(24,8)
molecules with queries of 4..20 nodes, a fifth of them perturbed; LogNormal(ln 24,0.45) molecules
with queries of 4..32 nodes, 30% with a ring), with odd sizes among them.

All results are whole numbers (offsets, query graph ids, match counts, hashes), so there is no
64-bit reference to give for them: equal inputs give equal outputs.  Pair lists go to result
arrays with room for every pair, which the program allocates once and hands to the C ABI (the
part past the pairs found stays zero).
"""
from __future__ import annotations

import ctypes
import functools

import numpy as np

from sigmo_amd import capi

# Molecule sequences are prefix-stable (molecule i of a seed does not depend on how many are made),
# so a run of molecules is cut from one longer run that is made once per process.
POOL_SEED = 1
POOL = {"normal": 200_000, "lognormal": 1_250_000}
DIST = {"normal": capi.SIZE_NORMAL, "lognormal": capi.SIZE_LOGNORMAL}
MEAN_NODES = {"normal": 24.0, "lognormal": 26.5}
# share of the (query graph, molecule) pairs that survive GMCR, for work()'s output bytes
SURVIVE = {"normal": 0.145, "lognormal": 0.08}


def listed():
    return [
        # the smoke test's size: one small search, bound by launches and the host round trip
        {"name": "batch_2k_x20", "kind": "batch", "molecules": 2_000, "sizes": "normal", "queries": 20, "kmin": 4, "kmax": 12,
         "R": 6, "first": True, "refresh": False, "result": "pairs"},
        # one substructure query over a mid-size library
        {"name": "batch_100k_x1", "kind": "batch", "molecules": 100_000, "sizes": "normal", "queries": 1, "kmin": 8, "kmax": 12,
         "R": 6, "first": True, "refresh": False, "result": "pairs"},
        # bench.py's config 1 step: database signatures recomputed, 100 queries, every pair read back
        {"name": "batch_100k_x100", "kind": "batch", "molecules": 100_000, "sizes": "normal", "queries": 100, "kmin": 4, "kmax": 20,
         "R": 6, "first": True, "refresh": True, "result": "pairs"},
        # counting every embedding, odd sizes, molecules of up to 128 nodes
        {"name": "batch_33331_x257_all", "kind": "batch", "molecules": 33_331, "sizes": "lognormal", "queries": 257, "kmin": 4,
         "kmax": 32, "R": 6, "first": False, "refresh": False, "result": "pairs"},
        # bench.py's config 2: 1 M molecules x 1,000 queries, answered per request of four queries
        {"name": "batch_1m_x1000", "kind": "batch", "molecules": 1_000_000, "sizes": "lognormal", "queries": 1000, "kmin": 4,
         "kmax": 32, "R": 6, "first": True, "refresh": False, "result": "requests"},
        # one request of the mean size (U[1,50] query graphs) through the online server, 1 M resident molecules
        {"name": "serve_1m_x25", "kind": "server", "molecules": 1_000_000, "sizes": "lognormal", "queries": 25, "kmin": 4, "kmax": 32,
         "R": 6, "first": True},
        # a burst of requests that arrive together and are batched
        {"name": "burst_300k_x12", "kind": "burst", "molecules": 300_000, "sizes": "lognormal", "requests": 12, "kmin": 4,
         "kmax": 32, "R": 6, "first": True},
        # the plain pipeline at the smoke test's size
        {"name": "plain_2k_x20", "kind": "plain", "molecules": 2_000, "sizes": "normal", "queries": 20, "kmin": 4, "kmax": 12,
         "R": 6, "first": True},
        # the plain pipeline on config 1, as the reference's driver runs it
        {"name": "plain_100k_x100", "kind": "plain", "molecules": 100_000, "sizes": "normal", "queries": 100, "kmin": 4, "kmax": 20,
         "R": 6, "first": True},
        # the plain pipeline on config 2's distributions (molecules of more than 64 nodes, queries of more than 12)
        {"name": "plain_150k_x300", "kind": "plain", "molecules": 150_000, "sizes": "lognormal", "queries": 300, "kmin": 4,
         "kmax": 32, "R": 6, "first": True},
        # the per-phase calls one by one, with wildcard query labels and the edge-label join
        {"name": "phases_20011_x64", "kind": "phases", "molecules": 20_011, "sizes": "normal", "queries": 64, "kmin": 4, "kmax": 20,
         "R": 3, "first": True, "wild": 0.05},
        # one pass over a shard held in host memory, in chunks on three workers, every pair handed back
        {"name": "stream_300k_x300", "kind": "stream", "molecules": 300_000, "sizes": "lognormal", "queries": 300, "kmin": 8,
         "kmax": 32, "R": 6, "first": True, "chunk": 80_000, "form": "batched", "workers": 3},
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], spread over the logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["batch", "batch", "batch", "server", "burst", "plain", "plain", "phases", "stream"])
    sizes = rng.choice(["normal", "lognormal"])
    kmin = rng.choice([4, 4, 6, 8])
    kmax = rng.randint(max(kmin, 10), 20 if sizes == "normal" else 32)
    case = {"kind": kind, "sizes": sizes, "kmin": kmin, "kmax": kmax, "R": rng.choice([6, 6, 6, 1, 2, 3, 4, 5, 7, 8]),
            "first": rng.random() < 0.75}
    most = 150_000 if sizes == "normal" else 600_000
    if kind == "batch":
        m = _between(rng, 500, most)
        q = _between(rng, 1, max(1, min(1000, 120_000_000 // m)))
        case |= {"molecules": m, "queries": q, "refresh": rng.random() < 0.3,
                 "result": "pairs" if m * q <= 20_000_000 else "requests"}
    elif kind == "server":
        case |= {"molecules": _between(rng, 5_000, most), "queries": rng.randint(1, 50)}
    elif kind == "burst":
        case |= {"molecules": _between(rng, 5_000, min(most, 300_000)), "requests": rng.randint(2, 16)}
    elif kind == "plain":
        m = _between(rng, 500, 150_000)
        case |= {"molecules": m, "queries": _between(rng, 1, max(1, min(400, 40_000_000 // m)))}
    elif kind == "phases":
        m = _between(rng, 300, 40_000)
        case |= {"molecules": m, "queries": _between(rng, 1, max(1, min(200, 2_000_000 // m))), "R": rng.randint(0, 6),
                 "wild": rng.choice([0.0, 0.05])}
    else:
        m = _between(rng, 20_000, min(most, 300_000))
        case |= {"molecules": m, "queries": _between(rng, 20, 300), "kmin": 8, "kmax": max(kmax, 12),
                 "chunk": max(5_000, m // rng.randint(2, 6)), "form": rng.choice(["batched", "batched", "plain"]),
                 "workers": rng.randint(1, 3)}
        if case["form"] == "plain":
            case["queries"] = min(case["queries"], 100)
    return case


@functools.lru_cache(maxsize=None)
def _pool(sizes):
    return capi.HostGraphs.molecules(POOL_SEED, POOL[sizes], DIST[sizes])


def _molecules(case, seed):
    pool, n = _pool(case["sizes"]), case["molecules"]
    return pool.slice(int(np.random.RandomState(seed % (1 << 32)).randint(0, pool.num_graphs - n + 1)), n)


def _queries(case, seed, count):
    normal = case["sizes"] == "normal"
    return capi.HostGraphs.queries(seed, count, case["kmin"], case["kmax"], DIST[case["sizes"]],
                                   perturb_frac=0.2 if normal else 0.0, ring_frac=-1.0 if normal else 0.3)


def _wild(host, share, seed):
    """The same query graphs with a share of their node labels replaced by the wildcard."""
    a = host.arrays()
    lab = a["node_labels"]
    lab[np.random.RandomState(seed % (1 << 32)).random_sample(lab.size) < share] = 255
    return capi.HostGraphs.from_arrays(a["graph_offsets"], a["row_offsets"], a["column_indices"], lab, a["edge_labels"])


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "ctx": capi.Context(0)}
    dh = _molecules(case, seed)
    if kind == "stream":
        s["qd"] = capi.DeviceGraph(s["ctx"], _queries(case, seed, case["queries"]))
        s["stream"] = capi.Stream(s["ctx"], s["qd"], dh, case["chunk"], case["form"], case["R"], case["first"], True, case["workers"])
        s["out"] = _room(case)
        return s
    s["dd"] = capi.DeviceGraph(s["ctx"], dh)
    if kind in ("batch", "server", "burst"):
        s["db"] = capi.Database(s["ctx"], s["dd"], case["R"])
        s["batch"] = capi.Batch(s["ctx"], s["db"])
    if kind == "burst":
        per = np.random.RandomState(seed % (1 << 32)).randint(1, 51, case["requests"])
        s["offsets"] = np.concatenate([[0], np.cumsum(per)]).astype(np.uint32)
        s["qh"] = _queries(case, seed, int(s["offsets"][-1]))
        s["arrival"] = np.zeros(case["requests"])
    else:
        s["qh"] = _queries(case, seed, case["queries"])
    if kind == "server":
        s["server"] = capi.Server([s["batch"]], find_first=case["first"])
    elif kind in ("batch", "plain", "phases"):
        if case.get("wild"):
            s["qh"] = _wild(s["qh"], case["wild"], seed)
        s["qd"] = capi.DeviceGraph(s["ctx"], s["qh"])
        if kind == "batch":
            n = case["queries"]
            s["offsets"] = np.unique(np.append(np.arange(0, n, -(-n // 250)), n)).astype(np.uint32)
        elif kind == "plain":
            s["pipe"] = capi.Pipeline(s["ctx"], s["qd"], s["dd"])
        if kind == "phases":
            s["rows"] = np.zeros(32 * case["queries"], np.int32)
            s["cand"] = capi.Candidates(s["ctx"], s["qd"].total_nodes, s["dd"].total_nodes)
            s["gmcr"] = capi.GMCR(s["ctx"])
        if case.get("result") != "requests":
            s["out"] = _room(case)
    s["ctx"].sync()
    return s


def _room(case):
    """Result arrays: GMCR offsets, and query graph ids and match counts with room for every pair."""
    pairs = case["molecules"] * case["queries"]
    return [np.zeros(case["molecules"] + 1, np.int32), np.zeros(pairs, np.int32), np.zeros(pairs, np.int32)]


def _totals(r):
    return [r["num_matches"], r["matched_pairs"], r["gmcr_pairs"]]


def _ptr(a, at=0):
    return ctypes.c_void_p(a.ctypes.data + 4 * at)


def _pairs(call, handle, s, pairs):
    off, idx, cnt = s["out"]
    capi.check(call(handle, _ptr(off), off.size, _ptr(idx) if pairs else None, _ptr(cnt) if pairs else None, pairs))
    return s["out"]


def _pass(s):
    """One pass of the stream, each chunk's pairs copied behind those of the chunks before it."""
    off, idx, cnt = s["out"]
    done = [0]

    def chunk(_user, _chunk, first, n, o, i, c, pairs):
        at = done[0]
        np.add(np.ctypeslib.as_array(o, (n + 1,))[1:].view(np.int32), at, out=off[first + 1:first + 1 + n])
        if pairs:
            ctypes.memmove(_ptr(idx, at), i, 4 * pairs)
            ctypes.memmove(_ptr(cnt, at), c, 4 * pairs)
        done[0] = at + pairs
        return 0

    r = capi.StreamResult()
    capi.check(capi.lib().sigmo_stream_pass(s["stream"]._h, capi.STREAM_CHUNK_FN(chunk), None, ctypes.byref(r)))
    return [r.num_matches, r.matched_pairs, r.gmcr_pairs] + s["out"]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "batch":
        if case["refresh"]:
            s["db"].refresh()
        out = _totals(s["batch"].run(s["qd"], case["first"]))
        if case["result"] == "pairs":
            return out + _pairs(capi.lib().sigmo_batch_pairs, s["batch"]._h, s, out[2])
        stats = s["batch"].request_stats(s["offsets"])
        return out + [np.array([(r["matched_pairs"], r["embeddings"], r["hash"]) for r in stats], np.uint64).view(np.int64)]
    if kind == "server":
        r = s["server"].poll(s["server"].submit(s["qh"]))
        return [r["status"], r["matched_pairs"], r["embeddings"], np.array([r["hash"]], np.uint64).view(np.int64)]
    if kind == "burst":
        r = capi.serve([s["batch"]], s["qh"], s["offsets"], s["arrival"], find_first=case["first"])
        return [r["status"], r["matched_pairs"], r["embeddings"], r["hash"].view(np.int64)]
    if kind == "plain":
        out = _totals(s["pipe"].execute(case["R"], case["first"]))
        return out + _pairs(capi.lib().sigmo_pipeline_pairs, s["pipe"]._h, s, out[2])
    if kind == "stream":
        return _pass(s)
    ctx, qd, dd, cand, gmcr = (s[x] for x in ("ctx", "qd", "dd", "cand", "gmcr"))
    sig = capi.Signature(ctx, dd.total_nodes, qd.total_nodes)  # signatures accumulate: each search starts from new ones
    sig.generate_data(dd)
    sig.generate_query(qd)
    capi.filter_candidates(ctx, qd, dd, sig, cand)
    for r in range(1, case["R"] + 1):
        sig.refine_data(dd, r)
        sig.refine_query(qd, r)
        capi.refine_candidates(ctx, qd, dd, sig, cand)
    gmcr.generate(qd, dd, cand)
    total, counts = capi.join_wildcard(ctx, qd, dd, cand, gmcr, case["first"])
    off, idx = gmcr.download()
    s["out"][0][:], s["out"][1][:idx.size], s["out"][2][:idx.size], s["rows"][:qd.total_nodes] = off, idx, counts, cand.counts()
    return [total, s["rows"]] + s["out"]


def work(case):
    """Inputs read once and results written once.  The batched form's input is its database (a
    label and R packed signatures of 8 bytes per node), the other kinds' the molecules' CSR
    arrays (about 4.2 + 2.1 x 5 bytes per node and its edges); results are 8 bytes per surviving
    pair plus the offsets, or 24 bytes per request."""
    kind, sizes = case["kind"], case["sizes"]
    nodes = case["molecules"] * MEAN_NODES[sizes]
    queries = case["requests"] * 25.5 if kind == "burst" else case["queries"]
    csr = nodes * (5.0 + 2.1 * 5.0)
    if kind in ("batch", "server", "burst"):
        read = nodes * (1.0 + 8.0 * case["R"]) + (csr if case.get("refresh") else 0.0)
    else:
        read = csr
    pairs = SURVIVE[sizes] * case["molecules"] * queries
    if kind in ("server", "burst") or case.get("result") == "requests":
        wrote = 24.0 * min(250.0, queries)
    else:
        wrote = 8.0 * pairs + 4.0 * case["molecules"]
    return {"bytes": read + wrote, "flops": 0.0}
