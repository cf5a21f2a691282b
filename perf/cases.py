"""Performance cases of the subgraph enumeration engine.

Every case is one call (or, for the server, one burst of calls) that a
user's program makes through the public Python entry points, on a graph that
is already resident: a fresh seeded graph per seed, uploaded by prepare().
Outputs are the counts, level outputs, per-member counts and match lists the
call returns, all of them integers.

A case is a dict of plain values:
  call    count    Device.count          count with level outputs
          total    Device.count_only     count alone (bench's house, 5-clique)
          range    Device.count          over a range of start vertices
          buckets  Device.count_buckets  packed member graphs, one count each
          list     Device.list_matches   match list of a GPSM plan
          serve    Server.submit / wait  a burst of pattern-count requests
  graph   rmat (scale, ef), er (n, m), or pack (members, nmin, nmax, dmin, dmax)
  query   Q0 .. Q13 (the pattern), algo (4 GPSM, 5 GPSM_REUSE, 6 LIGHT)
  ranked  keep the degree-ranked copy;  hubs  adjacency bitmaps from degree 256
  lane    lane_path_max and batch_mib  batch_bytes of the schedule (0: default)
"""
import functools
import random

import numpy as np
import torch

import subgraphmatchgpu_amd as sme

SQUARE_SCHEDULE = {"lane": 128, "batch_mib": 1024}  # what the autotuner picks for packed members
SERVE_WEIGHTS = ((0, 0.3), (1, 0.2), (2, 0.2), (3, 0.15), (4, 0.1), (7, 0.05))
ROWS_MAX = 1 << 20  # match-list cap, the default of Device.list_matches


def _rmat(scale, ef):
    return {"graph": "rmat", "scale": scale, "ef": ef}


def _er(n, m):
    return {"graph": "er", "n": n, "m": m}


def _pack(members, nmin, nmax, dmin, dmax):
    return {"graph": "pack", "members": members, "nmin": nmin, "nmax": nmax, "dmin": dmin, "dmax": dmax}


def _case(call, graph, query, algo=6, ranked=False, hubs=False, **more):
    return {"call": call, "query": query, "algo": algo, "ranked": ranked, "hubs": hubs, **graph, **more}


def listed():
    return [
        # the smallest call: a small sparse graph's triangles, where launches and latency count
        {"name": "er_300_triangle", **_case("count", _er(300, 1300), 0)},
        # R-MAT scale 14, triangle with level outputs, engine defaults
        {"name": "rmat14_triangle", **_case("count", _rmat(14, 16), 0)},
        # the headline pair: R-MAT scale 20, 4-clique and diamond, ranked copy and hub bitmaps
        {"name": "rmat20_clique4", **_case("count", _rmat(20, 16), 3, ranked=True, hubs=True)},
        {"name": "rmat20_diamond", **_case("count", _rmat(20, 16), 2, ranked=True, hubs=True)},
        # the large-graph pair (5-clique and house at edge factor 32), at the scales a pass of
        # at most a second or two allows
        {"name": "rmat19_clique5", **_case("count", _rmat(19, 32), 7, ranked=True)},
        {"name": "rmat19_house", **_case("total", _rmat(19, 32), 4, ranked=True)},
        # many packed Erdos-Renyi members, one count per member: triangle on the default
        # schedule, 4-cycle on the schedule the autotuner picks
        {"name": "pack_triangle", **_case("buckets", _pack(1000, 64, 8192, 4, 48), 0)},
        {"name": "pack_square", **_case("buckets", _pack(300, 64, 8192, 4, 48), 1, **SQUARE_SCHEDULE)},
        # a burst of requests (the service's pattern mix, random start ranges) over a resident graph
        {"name": "rmat16_serve", **_case("serve", _rmat(16, 16), -1, hubs=True, requests=40)},
        # one request alone: the house over a range of start vertices, original ids, with levels
        {"name": "rmat14_house_range", **_case("range", _rmat(14, 15), 4, hubs=True, first=0.21, share=0.33)},
        # a pattern with two unmaterialized vertices through every level of the engine
        {"name": "rmat13_near5clique", **_case("count", _rmat(13, 16), 6)},
        # a match list: full materialization, rows in lexicographic order
        {"name": "rmat14_list_triangle", **_case("list", _rmat(14, 16), 0, algo=4)},
    ]


def _log_int(rng, lo, hi):
    """Whole number spread over the logarithm of [lo, hi], odd two times in three."""
    v = int(round(lo * (hi / lo) ** rng.random()))
    return min(hi, max(lo, v | 1 if rng.random() < 2 / 3 else v))


def draw(rng):
    """One more case: one of the listed uses at other sizes, densities and options."""
    use = rng.choice(("small", "config", "clique", "house", "pack", "serve", "range", "pattern", "list"))
    ef = rng.randint(6, 20)
    if use == "small":
        n = _log_int(rng, 65, 4095)
        return _case("count", _er(n, n * rng.randint(2, min(24, n // 4))), rng.choice((0, 1, 2, 3)))
    if use == "config":
        on = rng.random() < 0.7
        return _case("count", _rmat(rng.randint(14, 20), ef), rng.choice((0, 2, 3)), ranked=on, hubs=on)
    if use == "clique":
        return _case(rng.choice(("count", "total")), _rmat(rng.randint(13, 18), rng.randint(9, 32)),
                     rng.choice((3, 7)), ranked=True, hubs=rng.random() < 0.5)
    if use == "house":
        return _case("total", _rmat(rng.randint(13, 18), rng.randint(9, 32)), 4, ranked=rng.random() < 0.8)
    if use == "pack":
        q = rng.choice((0, 1))
        nmax = _log_int(rng, 1000, 8192)
        graph = _pack(_log_int(rng, 20, 300), 64, nmax, 4, rng.randint(12, 48))
        return _case("buckets", graph, q, **(SQUARE_SCHEDULE if q and rng.random() < 0.7 else {}))
    if use == "serve":
        return _case("serve", _rmat(rng.randint(12, 15), ef), -1, hubs=True, requests=_log_int(rng, 5, 40))
    if use == "range":
        share = round(0.01 * 100 ** rng.random(), 4)
        return _case("range", _rmat(rng.randint(10, 14), ef), rng.choice((0, 1, 2, 3, 4)), hubs=rng.random() < 0.5,
                     first=round(rng.random() * (1 - share), 4), share=share)
    if use == "pattern":
        return _case("count", _rmat(rng.randint(9, 12), ef), rng.choice((1, 5, 6, 8, 9, 10, 12)))
    return _case("list", _rmat(rng.randint(9, 14), ef), rng.choice((0, 3)), algo=rng.choice((4, 5)))


def _graph(case, seed):
    """(host graph, member offsets or None) of a case."""
    if case["graph"] == "rmat":
        return sme.gen_rmat(case["scale"], case["ef"], seed=seed), None
    if case["graph"] == "er":
        return sme.gen_er(case["n"], case["m"], seed=seed), None
    return sme.gen_er_batch(case["members"], (case["nmin"], case["nmax"]), (case["dmin"], case["dmax"]), seed=seed)


def _requests(case, n, seed):
    """The burst: pattern by weight, start range of 1-100% of the vertices at a random place."""
    rng = random.Random(seed)
    queries, weights = zip(*SERVE_WEIGHTS)
    out = []
    for _ in range(case["requests"]):
        q = rng.choices(queries, weights)[0]
        length = max(1, int(n * rng.uniform(0.01, 1.0)))
        begin = rng.randint(0, n - length)
        out.append((q, begin, begin + length))
    return out


def prepare(case, seed):
    """The resident graph with its plan and device handle, or the open server and its requests."""
    g, offs = _graph(case, seed)
    if case["call"] == "serve":
        server = sme.Server(g, mem_cap_bytes=16 << 30, slots=4, hub_min_degree=256, hub_max_bytes=1 << 30)
        return {"call": "serve", "server": server, "requests": _requests(case, g.n, seed)}
    dev = sme.Device(0, budget_bytes=(16 if case["graph"] != "er" else 1) << 30)
    if case["hubs"]:
        dev.set_hub_bitmaps(256, 8 << 30)
    if case["ranked"]:
        dev.set_rank_order(True)
    if case.get("lane"):
        dev.set_tuning(lane_path_max=case["lane"], batch_bytes=case["batch_mib"] << 20, super_chunks=4)
    state = {"call": case["call"], "dev": dev, "graph": dev.upload(g), "plan": sme.Plan(case["query"], case["algo"])}
    if case["call"] == "range":
        state["begin"] = int(case["first"] * g.n)
        state["end"] = min(g.n, state["begin"] + max(1, int(case["share"] * g.n)))
    if offs is not None:
        state["bounds"] = offs.astype(np.uint32)
    return state


def run(state):
    """One pass; its counts, level outputs, per-member counts or match rows."""
    call = state["call"]
    if call == "serve":
        server = state["server"]
        ids = [server.submit(q, begin, end) for q, begin, end in state["requests"]]
        return np.array([server.wait(i)[0] for i in ids], dtype=np.int64)
    dev, graph, plan = state["dev"], state["graph"], state["plan"]
    if call == "list":
        rows, total = dev.list_matches(graph, plan, max_matches=ROWS_MAX)
        return {"rows": rows.view(np.int32), "total": total}
    if call == "buckets":
        counts, whole = dev.count_buckets(graph, plan, state["bounds"])
        return {"counts": counts.view(np.int64), "total": whole.count, "levels": np.array(whole.levels, dtype=np.int64)}
    if call == "range":
        got = dev.count(graph, plan, state["begin"], state["end"])
    elif call == "total":
        return {"count": dev.count_only(graph, plan).count}
    else:
        got = dev.count(graph, plan)
    return {"count": got.count, "levels": np.array(got.levels, dtype=np.int64)}


@functools.lru_cache(maxsize=None)
def _size(key):
    g, _ = _graph(dict(key), 1)
    return g.n, g.nnz


def work(case):
    """The resident graph read once (offsets and adjacency) and the outputs written once.  Counting is
    integer work: no floating operations."""
    key = tuple(sorted((k, case[k]) for k in case if k in ("graph", "scale", "ef", "n", "m", "members", "nmin", "nmax",
                                                          "dmin", "dmax")))
    n, nnz = _size(key)
    out = 8 * (case.get("requests") or case.get("members") or 1)
    if case["call"] == "list":
        out = ROWS_MAX * 4 * (3 if case["query"] == 0 else 4)
    return {"bytes": 8.0 * (n + 1) + 4.0 * nnz + out, "flops": 0.0}


def exact(case, seed):
    """Triangles, 4-cycles, diamonds and 4-cliques of a small graph from dense products of its adjacency
    matrix in 64 bits; None for the rest (all outputs are whole numbers)."""
    if case["graph"] != "er" or case["call"] != "count" or case["query"] > 3:
        return None
    g, _ = _graph(case, seed)
    rows = np.repeat(np.arange(g.n), np.diff(g.row_ptrs.astype(np.int64)))
    a = torch.zeros(g.n, g.n, dtype=torch.float64)
    a[torch.from_numpy(rows), torch.from_numpy(g.cols.astype(np.int64))] = 1.0
    if case["query"] == 1:  # pairs of common neighbours of each pair of opposite vertices, twice over
        c = a @ a
        c.fill_diagonal_(0.0)
        count = float((c * (c - 1)).sum()) / 8
    elif case["query"] == 3:
        up = torch.triu(a)
        count = 0.0
        for v in range(g.n):
            nb = torch.nonzero(up[v]).flatten()
            s = up[nb][:, nb]
            count += float(((s @ s) * s).sum())
    else:
        t = (a @ a) * a
        count = float(t.sum()) / 6 if case["query"] == 0 else float((t * (t - 1)).sum()) / 4
    return {"count": int(round(count)), "levels": None}
