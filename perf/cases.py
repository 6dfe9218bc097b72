"""The mining work whose speed is tracked, as callable cases.

``listed()`` names the cases, ``draw(rng)`` gives one more of the same
ranges, ``prepare(case, seed)`` builds what a user's program holds before the
call (a database resident on the GPU, a batch, a set of query codes), and
``run(state)`` is one pass through the public entry points.

Kinds of work (``case["kind"]``):

  mine     one database mined whole: ``mine(db, minsup)``.  With
           ``listing`` every pattern comes back (code, support, |Proj|), as a
           pattern sink of the driver sees them; without it the run counts,
           as ``graph_counting_output`` does, which is the mining driver's
           default when no output file is named.
  batch    several databases of different sizes and supports mined in one
           schedule from a resident ``Batch`` (counting).
  subsets  the server's mining request: a subset of a resident database is
           gathered into a ``Batch`` and mined, the patterns come back, the
           batch is closed.  The handle is new on every pass, as there.
  query    the server's other request: supports of pattern queries over a
           resident database, one at a time or many in one projection.

The databases come from the seeded generators with the sizes, label
alphabets and supports of the benchmark workloads, and odd sizes around them.
Every output is a whole number (patterns, supports, embedding counts) that
two correct programs agree on exactly.
"""
from __future__ import annotations

import math
import random

import numpy as np

import gpu_graph_mining_amd as gm
from gpu_graph_mining_amd import serving
from gpu_graph_mining_amd.workloads import abs_support


def listed():
    return [
        # the smallest call: 1,000 small graphs, two short levels; what an
        # interactive user or a test waits for -- launches and round trips
        {"name": "random_1k", "kind": "mine", "gen": "random", "graphs": 1000, "vmin": 10, "vmax": 30,
         "vlabels": 5, "elabels": 3, "edge_factor": 1.2, "support": 0.10, "listing": True, "room": 128,
         "budget": 0},
        # one support query (6 edges) against the resident molecule database:
        # the server's most frequent request at a low rate, a latency
        {"name": "query_one", "kind": "query", "gen": "molecule", "graphs": 50000, "queries": 1,
         "min_edges": 6, "max_edges": 6},
        # the server's query batch under load: 64 random-walk subgraphs of
        # 3-12 edges in one projection
        {"name": "query_64", "kind": "query", "gen": "molecule", "graphs": 50000, "queries": 64,
         "min_edges": 3, "max_edges": 12},
        # the server's mining request: 5,000 of the resident molecules at
        # 20 %, gathered, mined and listed through a handle of its own
        {"name": "subset_5k", "kind": "subsets", "gen": "molecule", "graphs": 50000, "subset": 5000,
         "support": 0.20, "room": 1024},
        # a ragged database of an odd size, graphs of 10 to 60 vertices
        {"name": "random_20k", "kind": "mine", "gen": "random", "graphs": 19997, "vmin": 10, "vmax": 60,
         "vlabels": 5, "elabels": 3, "edge_factor": 1.2, "support": 0.05, "listing": True, "room": 2048,
         "budget": 0},
        # transactions at the usual 5 %: more levels, a few thousand patterns
        {"name": "planted_10k", "kind": "mine", "gen": "planted", "graphs": 10000, "support": 0.05,
         "listing": False, "budget": 0},
        # the same kind of database under a memory budget: levels in pieces
        {"name": "planted_30k_budget", "kind": "mine", "gen": "planted", "graphs": 30011, "support": 0.05,
         "listing": False, "budget": 64 << 20},
        # molecules, rich in symmetric patterns, every pattern listed
        {"name": "molecule_50k", "kind": "mine", "gen": "molecule", "graphs": 50000, "support": 0.20,
         "listing": True, "room": 1024, "budget": 0},
        # many labels and graphs of up to 256 vertices: wide key spaces,
        # a root level of thousands of edges, no path masks
        {"name": "labels_40x6", "kind": "mine", "gen": "random", "graphs": 3001, "vmin": 100, "vmax": 256,
         "vlabels": 40, "elabels": 6, "edge_factor": 1.1, "support": 0.02, "listing": False, "budget": 0},
        # few, frequent patterns over the large transaction database
        {"name": "planted_100k_top", "kind": "mine", "gen": "planted", "graphs": 100000, "support": 0.20,
         "listing": True, "room": 1024, "budget": 0},
        # many databases of 200 to 20,000 graphs at 2-20 % in one schedule
        {"name": "batch_64", "kind": "batch", "jobs": 64, "min_graphs": 200, "max_graphs": 20000},
        # the largest: 100,000 transactions at 1 %, tens of thousands of
        # patterns -- the benchmark's headline workload
        {"name": "planted_100k", "kind": "mine", "gen": "planted", "graphs": 100000, "support": 0.01,
         "listing": False, "budget": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["random", "planted", "planted", "molecule", "labels", "batch", "subsets", "query"])
    if what == "random":
        vmin = rng.randint(8, 30)
        return {"kind": "mine", "gen": "random", "graphs": _log_int(rng, 500, 30000), "vmin": vmin,
                "vmax": vmin + rng.randint(0, 40), "vlabels": rng.randint(3, 8), "elabels": rng.randint(1, 4),
                "edge_factor": round(rng.uniform(1.0, 1.4), 2), "support": round(rng.uniform(0.05, 0.2), 3),
                "listing": rng.random() < 0.5, "room": 4096, "budget": 0}
    if what == "planted":
        support = round(math.exp(rng.uniform(math.log(0.02), math.log(0.3))), 3)
        return {"kind": "mine", "gen": "planted", "graphs": _log_int(rng, 1000, 60000), "support": support,
                "listing": support >= 0.1, "room": 4096, "budget": rng.choice([0, 0, 0, 128 << 20])}
    if what == "molecule":
        return {"kind": "mine", "gen": "molecule", "graphs": _log_int(rng, 300, 50000),
                "support": round(rng.uniform(0.1, 0.3), 3), "listing": rng.random() < 0.5, "room": 4096, "budget": 0}
    if what == "labels":
        return {"kind": "mine", "gen": "random", "graphs": _log_int(rng, 200, 4000), "vmin": 50,
                "vmax": rng.randint(60, 256), "vlabels": rng.randint(12, 60), "elabels": rng.randint(2, 8),
                "edge_factor": round(rng.uniform(1.0, 1.2), 2), "support": round(rng.uniform(0.02, 0.1), 3),
                "listing": False, "budget": 0}
    if what == "batch":
        return {"kind": "batch", "jobs": rng.randint(2, 48), "min_graphs": rng.randint(100, 400),
                "max_graphs": _log_int(rng, 1000, 20000)}
    graphs = _log_int(rng, 5000, 50000)
    if what == "subsets":
        return {"kind": "subsets", "gen": "molecule", "graphs": graphs,
                "subset": rng.randint(1000, min(10000, graphs)), "support": round(rng.uniform(0.1, 0.2), 3),
                "room": 4096}
    lo = rng.randint(3, 8)
    return {"kind": "query", "gen": "molecule", "graphs": graphs, "queries": _log_int(rng, 1, 64),
            "min_edges": lo, "max_edges": rng.randint(lo, 12)}


def _database(case, seed):
    if case["gen"] == "random":
        return gm.GraphDB.random(seed, case["graphs"], case["vmin"], case["vmax"], case["edge_factor"],
                                 case["vlabels"], case["elabels"])
    if case["gen"] == "planted":
        return gm.GraphDB.planted(seed, case["graphs"])
    return gm.GraphDB.molecule(seed, case["graphs"])


def prepare(case, seed):
    kind = case["kind"]
    rng = random.Random(seed)
    if kind == "batch":
        lo, hi = math.log(case["min_graphs"]), math.log(case["max_graphs"])
        dbs, mins = [], []
        for _ in range(case["jobs"]):
            n = int(round(math.exp(rng.uniform(lo, hi))))
            dbs.append(gm.GraphDB.random(rng.getrandbits(63), n, 10, 60, 1.2, 5, 3))
            mins.append(abs_support(rng.uniform(0.02, 0.20), n))
        return {"kind": kind, "batch": gm.Batch(dbs), "mins": mins}
    db = _database(case, seed)
    db.upload()
    if kind == "query":
        arrays, codes = db.arrays(), []
        while len(codes) < case["queries"]:
            code = serving.random_walk_code(arrays, rng, rng.randint(case["min_edges"], case["max_edges"]))
            if code is not None:
                codes.append(code)
        return {"kind": kind, "db": db, "codes": codes}
    if kind == "subsets":
        ids = sorted(rng.sample(range(case["graphs"]), case["subset"]))
        return {"kind": kind, "db": db, "ids": ids, "minsup": abs_support(case["support"], case["subset"]),
                "room": case["room"]}
    return {"kind": kind, "db": db, "minsup": abs_support(case["support"], case["graphs"]),
            "listing": case["listing"], "room": case.get("room", 0), "budget": case["budget"]}


def _listing(patterns, room):
    """The patterns as arrays with room for `room` patterns of twelve edges
    on average (unused places hold -1): the tuples of all codes one after the
    other, the codes' lengths, supports and embedding counts."""
    tuples = [t for code, _, _ in patterns for t in code]
    rows = [(len(code), support, n) for code, support, n in patterns]
    codes = np.full((12 * room, 5), -1, dtype=np.int32)
    facts = np.full((room, 3), -1, dtype=np.int64)
    if rows:
        codes[:len(tuples)] = tuples
        facts[:len(rows)] = rows
    return {"codes": codes, "facts": facts}


def _counts(stats):
    return {k: int(stats[k]) for k in ("n_patterns", "e_child", "e_root", "e_cand")}


def run(state):
    kind = state["kind"]
    if kind == "query":
        return np.array(gm.support(state["db"], state["codes"]), dtype=np.int64)
    if kind == "batch":
        _, stats = state["batch"].mine(state["mins"], count_only=True)
        return _counts(stats)
    if kind == "subsets":
        batch = gm.Batch.from_subsets(state["db"], [state["ids"]])
        try:
            patterns, stats = batch.mine([state["minsup"]], collect_proj=True)
        finally:
            batch.close()
        return {**_listing(patterns[0], state["room"]), **_counts(stats)}
    patterns, stats = gm.mine(state["db"], state["minsup"], collect_proj=state["listing"],
                              count_only=not state["listing"], mem_budget=state["budget"])
    out = _counts(stats)
    return {**_listing(patterns, state["room"]), **out} if state["listing"] else out


def work(case):
    """The packed database read once (the path works on integers: no
    floating-point operations).  Means of the generators: a random graph has
    the middle of its vertex range, a planted one 30 edges on 26 vertices, a
    molecule 26 edges on 25 vertices."""
    def graphs_bytes(n, nv, ne):
        return n * (4 + nv * 5 + ne * 8)  # graph offset; vertex offset and label; two packed 4-byte entries an edge

    if case["kind"] == "batch":
        lo, hi = case["min_graphs"], case["max_graphs"]
        mean = (hi - lo) / math.log(hi / lo) if hi > lo else lo
        return {"bytes": case["jobs"] * graphs_bytes(mean, 35, 42), "flops": 0}
    if case["gen"] == "random":
        nv = (case["vmin"] + case["vmax"]) / 2
        return {"bytes": graphs_bytes(case["graphs"], nv, nv * case["edge_factor"]), "flops": 0}
    if case["gen"] == "planted":
        return {"bytes": graphs_bytes(case["graphs"], 26, 32), "flops": 0}
    return {"bytes": graphs_bytes(case["subset"] if case["kind"] == "subsets" else case["graphs"], 25, 26), "flops": 0}
