"""The compact level kernels (graphs of at most 64 vertices, small label
alphabets) at the edges of their layout, against the oracle: patterns,
supports, |Proj(P)|, E_child and E_cand, all whole numbers, exactly equal.

A vertex's neighbours come in groups of four, the first two of which are
tested in registers; a block is up to 64 rows of whole segments (rows of one
graph), longer segments are carried from block to block; a chunk's list names
rows up to 8,192 from a base; label pairs are tested in 32 bits below 32 of
them."""
import random

import pytest

import gpu_graph_mining_amd as gm
from oracle import py_oracle as po

pytestmark = pytest.mark.gpu


def star(leaves, vlab=0, elab=0):
    return [vlab] * (leaves + 1), [(0, v, elab) for v in range(1, leaves + 1)]


def clique(n, elab=0):
    return [0] * n, [(a, b, elab) for a in range(n) for b in range(a + 1, n)]


def paths(k):
    """k disjoint paths of three equal vertices: 4 k rows of the 1-edge
    pattern, 2 k of the path's."""
    return [0] * (3 * k), [e for i in range(k) for e in ((3 * i, 3 * i + 1, 0), (3 * i + 1, 3 * i + 2, 0))]


def tree(rng, n, nvl, nel, extra=0):
    labels = [rng.randrange(nvl) for _ in range(n)]
    pairs = {(rng.randrange(v), v) for v in range(1, n)}
    while extra:
        a, b = sorted(rng.sample(range(n), 2))
        extra -= (a, b) not in pairs
        pairs.add((a, b))
    return labels, [(a, b, rng.randrange(nel)) for a, b in sorted(pairs)]


def all_labels(nvl, nel):
    """A graph that holds every label, so that the alphabets have these sizes."""
    n = max(nvl, nel + 1)
    return [v % nvl for v in range(n)], [(v, v + 1, v % nel) for v in range(n - 1)]


def mixed(nvl, nel, sizes, extra=3):
    rng = random.Random(17 * nvl + nel)
    return [all_labels(nvl, nel)] + [tree(rng, n, nvl, nel, min(extra, n * (n - 1) // 2 - (n - 1))) for n in sizes]


CASES = {
    # one to four groups a vertex (4 | 5, 8 | 9 neighbours); segments of 11,880 rows
    "stars": ([star(n) for n in (1, 3, 4, 5, 8, 9, 12, 12)], 1, 4),
    # backward edges among a vertex's third group
    "cliques": ([clique(n) for n in (3, 5, 6, 9, 10)], 1, 3),
    # segments of exactly 64, 32, 60, 68, 84 and 4 rows, whole blocks of them
    "paths": ([paths(k) for k in (16, 16, 8, 8, 15, 17, 1, 21, 16)] + [paths(16)] * 9, 1, 0),
    # the largest graphs, two of them with 64 rows in one segment
    "64_vertices": (mixed(3, 2, [64, 64, 63, 64, 2, 1, 33]) + [star(63)], 1, 3),
    # 25 label pairs (32-bit masks), 31, and 42 and 56 (64-bit masks; 56 = 7 edge labels x 8, the largest keys)
    "labels_5x5": (mixed(5, 5, [20] * 40), 2, 4),
    "labels_31x1": (mixed(31, 1, [30] * 30), 2, 4),
    "labels_6x7": (mixed(6, 7, [25] * 40), 2, 4),
    "labels_8x7": (mixed(8, 7, [40] * 30), 2, 4),
    # one past the compact alphabets: the general kernels
    "labels_8x8": (mixed(8, 8, [40] * 30), 2, 4),
    # graphs without edges or vertices between the others
    "empty_graphs": ([([], []), star(3), ([0], []), clique(4), ([], []), star(3)], 1, 0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_compact_levels_match_the_oracle(name):
    graphs, minsup, max_edges = CASES[name]
    db = gm.GraphDB.from_graphs(graphs)
    opats, ost = po.mine_arrays(db.arrays(), minsup, max_edges=max_edges)
    want = {po.normalize(c): (s, n) for c, s, n in opats}
    print("case", name, len(want), "patterns", flush=True)
    for kw in ({}, {"path_pruning": False, "speculate": 2}, {"mem_budget": 20000}, {"canon_host": 2, "chunk_rows": 64}):
        if kw.get("mem_budget") and len(want) > 2000:
            continue  # (a level step per piece)
        print("options", kw, flush=True)
        pats, st = gm.mine(db, minsup, max_edges=max_edges, collect_proj=True, **kw)
        assert {po.normalize(c): (s, n) for c, s, n in pats} == want and len(pats) == len(want)
        assert (st["e_child"], st["e_cand"]) == (ost["e_child"], ost["e_cand"])


def test_subsets_of_a_compact_database():
    """Gathered groups and root rows: each subset's patterns are the oracle's
    on the same graphs, in a batch of several subsets (one of them empty)."""
    graphs = mixed(4, 3, [3, 9, 30, 17, 1, 25, 40, 12] * 6)
    db = gm.GraphDB.from_graphs(graphs)
    db.upload()
    rng = random.Random(3)
    subsets = [rng.sample(range(len(graphs)), 20), list(range(len(graphs))), [], [5, 5, 5], [0]]
    batch = gm.Batch.from_subsets(db, subsets)
    res, _ = batch.mine([4, 6, 1, 3, 1], collect_proj=True)
    for ids, minsup, pats in zip(subsets, [4, 6, 1, 3, 1], res):
        arrays = gm.GraphDB.from_graphs([graphs[i] for i in ids]).arrays() if ids else None
        opats = po.mine_arrays(arrays, minsup)[0] if ids else []
        assert {po.normalize(c): (s, n) for c, s, n in pats} == {po.normalize(c): (s, n) for c, s, n in opats}


@pytest.mark.parametrize("sink", [False, True])
def test_children_chosen_on_the_device(sink):
    """Levels of hundreds of keys, chosen on the device, with symmetric codes
    (stars of five and six equal leaves) that its check leaves to the host
    half way; with a sink, the patterns of every level are reported in key
    order, and a sink that stops the run is heard."""
    rng = random.Random(11)
    graphs = []
    for _ in range(30):
        labels, edges = tree(rng, 24, 3, 2, 3)
        n = len(labels)
        graphs.append((labels + [0] * 8, edges + [(n, n + i, 0) for i in range(1, 8)]))
    db = gm.GraphDB.from_graphs(graphs)
    opats, ost = po.mine_arrays(db.arrays(), 4, max_edges=6)
    want = {po.normalize(c): (s, n) for c, s, n in opats}
    print(len(want), "patterns", flush=True)
    if not sink:
        pats, st = gm.mine(db, 4, max_edges=6, collect_proj=True)
        assert {po.normalize(c): (s, n) for c, s, n in pats} == want and len(pats) == len(want)
        assert (st["e_child"], st["e_cand"]) == (ost["e_child"], ost["e_cand"])
        assert st["canon_host_keys"] > 0
        return
    seen = []
    gm.mine(db, 4, max_edges=6, on_pattern=lambda c, s, n: seen.append((c, s)))
    assert {po.normalize(c): s for c, s in seen} == {c: s for c, (s, _) in want.items()}
    assert [len(c) for c, _ in seen] == sorted(len(c) for c, _ in seen)
    for stop_at in (1, len(seen) // 2, len(seen)):
        got = []
        with pytest.raises(gm.GMError) as e:
            gm.mine(db, 4, max_edges=6, on_pattern=lambda c, s, n: (got.append((c, s)), len(got) < stop_at)[1])
        assert e.value.code == gm.GM_E_CALLBACK and got == seen[:stop_at]


@pytest.mark.parametrize("graphs,nvl,nel,minsup", [(40, 16, 8, 3), (40, 16, 9, 3), (40, 3, 2, 12), (6000, 3, 2, 2400),
                                                   (6000, 6, 1, 1500), (6000, 7, 5, 600)])
def test_reductions_of_few_and_many_counters(graphs, nvl, nel, minsup):
    """Root keys at and past the 2,048 that one workgroup reduces (general
    kernels, with item sums), and databases of enough chunks for counter
    replicas: patterns and counts equal those of the entry point whose buffers
    and kernels are the general ones with one replica, and the oracle's."""
    db = gm.GraphDB.random(graphs, graphs, 8, 14, 1.1, nvl, nel)
    db.upload()
    key = lambda pats: sorted((tuple(c), s, n) for c, s, n in pats)
    pats, st = gm.mine(db, minsup, collect_proj=True)
    other, so = gm.mine_noalloc(db, minsup, collect_proj=True)
    assert pats and key(pats) == key(other)
    assert all(st[k] == so[k] for k in ("n_patterns", "e_root", "e_child", "e_cand"))
    if graphs == 40:
        opats, ost = po.mine_arrays(db.arrays(), minsup)
        assert sorted((po.normalize(c), s, n) for c, s, n in pats) == sorted((c, s, n) for c, s, n in opats)
        assert (st["e_child"], st["e_cand"]) == (ost["e_child"], ost["e_cand"])


@pytest.mark.parametrize("graphs,nvl,nel,factor,minsup", [(12000, 3, 2, 1.4, 240), (12000, 2, 1, 1.7, 1800), (300, 3, 1, 1.6, 30)])
def test_extensions_infrequent_at_the_parent_are_not_listed(graphs, nvl, nel, factor, minsup):
    """The sibling rule drops only what cannot be frequent, forward and backward
    (cycles), with children chosen on the device (12,000 graphs) and on the
    host, checked there or written ahead, in pieces and by job: patterns,
    supports, |Proj| and E_cand are those of a run without path pruning."""
    db = gm.GraphDB.random(5, graphs, 6, 12, factor, nvl, nel)
    db.upload()
    key = lambda pats: sorted((tuple(c), s, n) for c, s, n in pats)
    want, so = gm.mine(db, minsup, collect_proj=True, path_pruning=False)
    assert any(t[0] > t[1] for c, _, _ in want for t in c) and so["pruned"] == 0
    for kw in ({}, {"canon_host": 1}, {"canon_host": 2}, {"speculate": 2}, {"mem_budget": 6 << 20}):
        print("options", kw, flush=True)
        pats, st = gm.mine(db, minsup, collect_proj=True, **kw)
        assert key(pats) == key(want)
        assert all(st[k] == so[k] for k in ("n_patterns", "e_root", "e_child", "e_cand"))
        assert st["pruned"] > 0
    ids = [list(range(0, graphs, 2)), list(range(graphs))]
    batch = gm.Batch.from_subsets(db, ids)
    res, _ = batch.mine([minsup, minsup], collect_proj=True)
    assert key(res[1]) == key(want)
    half = db.subset(ids[0])
    assert key(res[0]) == key(gm.mine(half, minsup, collect_proj=True, path_pruning=False)[0])
    batch.close()
