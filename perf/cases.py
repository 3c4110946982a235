"""What the performance of this library is measured on.

The cases are the calls that programs make: count one graph again and again,
count a graph that was just loaded, run one call over many graphs, serve a
stream of requests -- from graphs of a thousand vertices, where launches and
latency are all there is, to the triangle count of RMAT scale 22.  RMAT graphs have the quadrant probabilities 0.57/0.19/0.19/0.05;
"er" graphs are `draws` uniform pairs of `n` vertices (the control without
skew, with odd sizes).  Counts come back as uint64 arrays.
"""
from __future__ import annotations

import math
import random

import numpy as np

import mercury_amd as ma

_RMAT = (0.57, 0.19, 0.19)  # a, b, c
_MIX = ("TC", "P1", "P2", "P3", "P4", "P5", "P6", "P7", "P8")


def listed():
    return [
        # One small graph counted over and over by a program that holds it:
        # launches, the copy of the count and the wait are most of it.
        {"name": "tc_rmat10", "kind": "count", "pattern": "TC",
         "graph": "rmat", "scale": 10, "edge_factor": 16},
        # The plain triangle count of one ordinary graph.
        {"name": "tc_rmat16", "kind": "count", "pattern": "TC",
         "graph": "rmat", "scale": 16, "edge_factor": 16},
        # The headline: a large skewed graph, resident, counted repeatedly.
        {"name": "tc_rmat22", "kind": "count", "pattern": "TC",
         "graph": "rmat", "scale": 22, "edge_factor": 16},
        # The same size without skew: millions of tiny neighbour lists.
        {"name": "tc_er22", "kind": "count", "pattern": "TC",
         "graph": "er", "n": 1 << 22, "draws": 16 << 22},
        # What the tc_challenge program does after reading a file: upload
        # the CSR, orient and plan on the device, count once, free.
        {"name": "fresh_rmat20", "kind": "fresh",
         "graph": "rmat", "scale": 20, "edge_factor": 16},
        # Claws of a graph of odd size without skew, where triangles are few
        # and the passes over vertices and arcs are most of the work.
        {"name": "p1_er300k", "kind": "count", "pattern": "P1",
         "graph": "er", "n": 300_007, "draws": 2_400_011},
        # Induced paths on four vertices at the size of the pattern
        # configuration (P1, claws, runs the first part of the same work).
        {"name": "p4_rmat20", "kind": "count", "pattern": "P4",
         "graph": "rmat", "scale": 20, "edge_factor": 16},
        # The clique-based five-vertex patterns (P7; P8 runs the same).
        {"name": "p7_rmat18", "kind": "count", "pattern": "P7",
         "graph": "rmat", "scale": 18, "edge_factor": 16},
        # The other five-vertex patterns (P2, P3, P5 and P6 run the same
        # passes) on a large graph and on a small one.
        {"name": "p2_rmat18", "kind": "count", "pattern": "P2",
         "graph": "rmat", "scale": 18, "edge_factor": 16},
        {"name": "p6_rmat10", "kind": "count", "pattern": "P6",
         "graph": "rmat", "scale": 10, "edge_factor": 16},
        # Many graphs of uneven size in one call: TC, P2 and P4 of each.
        {"name": "batch_24", "kind": "batch", "graphs": 24, "lanes": 8,
         "low_scale": 10, "high_scale": 14},
        # A request stream on resident graphs, Poisson arrivals, patterns
        # drawn uniformly.
        {"name": "serve_64", "kind": "serve", "graphs": 8, "low_scale": 10,
         "high_scale": 14, "edge_factor": 16, "requests": 64,
         "rate": 2000.0},
    ]


def _log_int(rng: random.Random, low: float, high: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_graph(rng: random.Random, most: float) -> dict:
    """A graph of at most `most` draws, and hardly ever of a round size."""
    if rng.random() < 0.65:
        scale = rng.randint(8, int(math.log2(most / 4)))
        return {"graph": "rmat", "scale": scale,
                "edge_factor": _log_int(rng, 4, min(32, most / 2**scale))}
    n = _log_int(rng, 300, most / 12)
    return {"graph": "er", "n": n,
            "draws": min(int(most), int(n * rng.uniform(3, 24)))}


def draw(rng: random.Random) -> dict:
    kind = rng.choice(("tc", "tc", "p4", "p5", "p5", "fresh", "batch",
                       "serve"))
    if kind == "tc":
        return {"kind": "count", "pattern": "TC", **_draw_graph(rng, 2**25)}
    if kind == "p4":
        return {"kind": "count", "pattern": rng.choice(("P1", "P4")),
                **_draw_graph(rng, 2**22)}
    if kind == "p5":
        return {"kind": "count",
                "pattern": rng.choice(("P2", "P3", "P5", "P6", "P7", "P8")),
                **_draw_graph(rng, 2**20)}
    if kind == "fresh":
        return {"kind": "fresh", **_draw_graph(rng, 2**23)}
    low = rng.randint(8, 11)
    if kind == "batch":
        return {"kind": "batch", "graphs": rng.randint(5, 24),
                "lanes": rng.choice((1, 4, 8)), "low_scale": low,
                "high_scale": rng.randint(low + 1, 13)}
    return {"kind": "serve", "graphs": rng.randint(3, 12), "low_scale": low,
            "high_scale": rng.randint(low + 1, 13),
            "edge_factor": rng.randint(5, 16),
            "requests": rng.randint(20, 80),
            "rate": round(rng.uniform(500, 4000), 1)}


def _pool(case: dict) -> list:
    """The graphs of a batch or a server: scales spread evenly over the
    range, a batch's edge factors 4, 8, 16, 32 in turn."""
    k, low, high = case["graphs"], case["low_scale"], case["high_scale"]
    return [{"graph": "rmat",
             "scale": low + round((high - low) * i / max(k - 1, 1)),
             "edge_factor": case.get("edge_factor", (4, 8, 16, 32)[i % 4])}
            for i in range(k)]


def _graph(spec: dict, seed: int) -> ma.Graph:
    if spec["graph"] == "er":
        return ma.Graph.er(spec["n"], spec["draws"], seed)
    return ma.Graph.rmat(spec["scale"], spec["edge_factor"], *_RMAT,
                         seed=seed)


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    state = {"case": case}
    if kind == "count":
        g = _graph(case, seed)
        state["dg"] = ma.DeviceGraph(g, 0, device_plan=True)
        state["pattern"] = ma.PATTERN_NAMES[case["pattern"]]
    elif kind == "fresh":
        state["g"] = _graph(case, seed)
    elif kind == "batch":
        graphs = [_graph(s, 1000 * seed + i)
                  for i, s in enumerate(_pool(case))]
        dgs = [ma.DeviceGraph(g, 0) for g in graphs]
        state["batch"] = ma.Batch(0, lanes=case["lanes"])
        state["queries"] = [(dg, p) for dg in dgs
                            for p in (ma.TC, ma.P2, ma.P4)]
    else:
        server = ma.Server(0, slots=3, lanes=4)
        ids = [server.add_graph(_graph(s, 1000 * seed + i))
               for i, s in enumerate(_pool(case))]
        rng = random.Random(seed)
        at, schedule = 0.0, []
        for _ in range(case["requests"]):
            at += rng.expovariate(case["rate"]) * 1e6
            schedule.append((rng.choice(ids),
                             ma.PATTERN_NAMES[rng.choice(_MIX)], int(at)))
        state["server"], state["schedule"] = server, schedule
    return state


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "count":
        if state["pattern"] == ma.TC:
            count, _ = state["dg"].tc_count()
        else:
            count, _ = state["dg"].pattern_count(state["pattern"])
        return np.array([count], dtype=np.uint64)
    if kind == "fresh":
        dg = ma.DeviceGraph(state["g"], 0, device_plan=True)
        count, _ = dg.tc_count()
        dg.close()
        return np.array([count], dtype=np.uint64)
    if kind == "batch":
        counts, _ = state["batch"].run(state["queries"])
        return np.array(counts, dtype=np.uint64)
    done = state["server"].replay(state["schedule"])
    return {"counts": np.array([r.count for r in done], dtype=np.uint64),
            "status": np.array([r.status for r in done], dtype=np.int32)}


def _edges(spec: dict) -> tuple[int, float]:
    """Vertices and expected undirected edges of a graph."""
    if spec["graph"] == "er":
        n, draws = spec["n"], spec["draws"]
        pairs = n * (n - 1) / 2
        return n, -pairs * math.expm1(-draws * 2 / (n * n))
    # RMAT: cells by how often each quadrant is taken; b = c, so a pair and
    # its mirror are equally likely, and pairs off the diagonal count once.
    s, (a, b, _) = spec["scale"], _RMAT
    d = 1 - a - 2 * b
    draws = spec["edge_factor"] << s
    m = 0.0
    for k in range(1, s + 1):  # k levels in the off-diagonal quadrants
        for i in range(s - k + 1):
            cells = math.comb(s, k) * math.comb(s - k, i) * 2.0**k
            p = a**i * d**(s - k - i) * b**k
            m -= cells / 2 * math.expm1(-2 * p * draws)
    return 1 << s, m


def work(case: dict) -> dict:
    """Bytes of one pass: a resident graph's edges once each (4 bytes) and
    its row pointers, or the host CSR (both directions of each edge) of a
    graph that is uploaded.  The set intersections compare integers; there
    is no floating-point work."""
    kind = case["kind"]
    if kind == "batch":
        return {"bytes": sum(work({"kind": "count", **s})["bytes"]
                             for s in _pool(case)), "flops": 0}
    if kind == "serve":
        pool = sum(work({"kind": "count", **s})["bytes"]
                   for s in _pool(case))
        return {"bytes": pool, "flops": 0}
    n, m = _edges(case)
    return {"bytes": 8 * (n + 1) + (8 if kind == "fresh" else 4) * m,
            "flops": 0}


def _dag(rowptr, col):
    """The DAG by (degree, id): row pointers, columns, the row of each."""
    deg = np.diff(rowptr)
    src = np.repeat(np.arange(len(deg)), deg)
    keep = (deg[col] > deg[src]) | ((deg[col] == deg[src]) & (col > src))
    out = np.bincount(src[keep], minlength=len(deg))
    return np.concatenate([[0], np.cumsum(out)]), col[keep], src[keep]


def _triangles(rowptr, col) -> int | None:
    """Wedges of the DAG closed by an arc, looked up in the sorted arcs."""
    n = len(rowptr) - 1
    drp, dcol, dsrc = _dag(rowptr, col)
    out = np.diff(drp)
    lens = out[dcol]
    if int(lens.sum()) > 60_000_000:
        return None
    key = dsrc * np.int64(n) + dcol
    total = 0
    for b in range(0, len(dcol), 1 << 20):
        ln = lens[b:b + (1 << 20)]
        u = np.repeat(dsrc[b:b + (1 << 20)], ln)
        first = np.repeat(drp[dcol[b:b + (1 << 20)]], ln)
        off = np.arange(len(u)) - np.repeat(np.cumsum(ln) - ln, ln)
        want = u * np.int64(n) + dcol[first + off]
        at = np.searchsorted(key, want)
        at[at == len(key)] = 0
        total += int(np.count_nonzero(key[at] == want)) if len(key) else 0
    return total


def exact(case: dict, seed: int):
    """Triangle counts of the graphs that numpy counts in seconds; the
    other outputs are whole numbers that numpy would take minutes for."""
    kind = case["kind"]
    if kind not in ("count", "fresh") or case.get("pattern", "TC") != "TC":
        return None
    if _edges(case)[1] > 3e6:
        return None
    rowptr, col = _graph(case, seed).csr()
    count = _triangles(rowptr, col.astype(np.int64))
    return None if count is None else np.array([count], dtype=np.uint64)
