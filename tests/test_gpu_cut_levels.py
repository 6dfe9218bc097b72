"""Levels that do not go through in one piece or at the first try.

Levels cut into pieces without a memory budget (more counter keys than a
level step takes, GraphDB.set_limits), on compact databases: a piece's
children, chosen on the device, and their children are mined while the cut
level's rows wait for its next piece.  Patterns, supports, |Proj(P)|, E_child
and E_cand are the oracle's, for one database and for the jobs of a batch.  Levels whose candidate lists
outgrow their pool (set small here) are listed again into a larger one, with
the same results."""
import random
import re

import pytest

import gpu_graph_mining_amd as gm
from oracle import py_oracle as po

from test_gpu_compact import all_labels, clique, star, tree

pytestmark = pytest.mark.gpu


def _key(pats):
    return sorted((po.normalize(c), s, n) for c, s, n in pats)


def _chosen_under_a_cut_level(trace):
    """Levels whose children the device chose while an earlier level had
    pieces to come."""
    cut, n = set(), 0
    for line in trace.splitlines():
        level = int(re.search(r"^\[gm level (\d+)\]", line)[1])
        cut = {x for x in cut if x < level}
        piece = re.search(r"piece \d+-(\d+) of (\d+)", line)
        if piece and int(piece[1]) < int(piece[2]):
            cut.add(level)
        elif not piece and cut and int(re.search(r"children (\d+)", line)[1]):
            n += 1
    return n


@pytest.fixture
def trace(monkeypatch, capfd):
    monkeypatch.setenv("GM_LEVEL_TRACE", "1")

    def read():
        return capfd.readouterr().err

    return read


@pytest.mark.parametrize("piece_keys", [8000, 16000, 64000])
def test_a_cut_level_keeps_its_rows(trace, piece_keys):
    db = gm.GraphDB.molecule(3, 100)
    opats, ost = po.mine_arrays(db.arrays(), 4, max_edges=8)
    db.set_limits(piece_keys=piece_keys)
    trace()
    pats, st = gm.mine(db, 4, max_edges=8, collect_proj=True)
    assert _chosen_under_a_cut_level(trace()) > 0
    assert _key(pats) == _key(opats)
    assert (st["e_child"], st["e_cand"]) == (ost["e_child"], ost["e_cand"])


def test_a_cut_level_of_a_batch_keeps_its_rows(trace):
    db = gm.GraphDB.molecule(3, 100)
    jobs = [(list(range(100)), 8), (list(range(1, 100, 2)), 5), (list(range(30)), 6)]
    batch = gm.Batch.from_subsets(db, [ids for ids, _ in jobs])
    batch.set_limits(piece_keys=16000)
    trace()
    res, _ = batch.mine([minsup for _, minsup in jobs], collect_proj=True)
    assert _chosen_under_a_cut_level(trace()) > 0
    for (ids, minsup), pats in zip(jobs, res):
        assert _key(pats) == _key(po.mine_arrays(db.subset(ids).arrays(), minsup)[0])
    batch.close()
    # a batch that takes over the buffers has the default limits again
    batch = gm.Batch.from_subsets(db, [ids for ids, _ in jobs])
    assert [_key(pats) for pats in batch.mine([minsup for _, minsup in jobs], collect_proj=True)[0]] == [_key(p) for p in res]
    assert not re.search(r"piece 0-(?!(\d+) of \1 )", trace())
    batch.close()


@pytest.mark.parametrize("limits", [(-1, 0), ((1 << 26) + 1, 0), (0, -1)])
def test_limits_outside_their_range_are_refused(limits):
    db = gm.GraphDB.molecule(3, 5)
    with pytest.raises(gm.GMError) as e:
        db.set_limits(*limits)
    assert e.value.code == gm.GM_E_ARG


def test_the_path_table_is_the_root_pieces_own(trace):
    """A root level cut by jobs: the first piece's 2-edge level is chosen on the
    device, the second piece's (few edges) on the host and its 3-edge level on
    the device again, which takes the second piece's 2-edge paths."""
    rng = random.Random(5)
    rich = [gm.GraphDB.from_graphs([all_labels(3, 2)] + [tree(rng, 16, 3, 2, 2) for _ in range(12)]) for _ in range(7)]
    single = gm.GraphDB.from_graphs([([0, 0], [(0, 1, 0)])])
    # 18 root keys a job: 222 jobs in the first piece
    dbs = rich[:6] + [single] * 220 + rich[6:]
    minsups = [4] * 6 + [2] * 220 + [2]
    batch = gm.Batch(dbs)
    batch.set_limits(piece_keys=4000)
    trace()
    res, _ = batch.mine(minsups, collect_proj=True)
    lines = trace().splitlines()
    second = [i for i, line in enumerate(lines) if line.startswith("[gm level 0]")][1]
    assert any(line.startswith("[gm level 1] device-chosen") for line in lines[:second])
    assert lines[second + 1].startswith("[gm level 1] piece")
    assert lines[second + 2].startswith("[gm level 2] device-chosen")
    for i, (db, minsup, pats) in enumerate(zip(dbs, minsups, res)):
        assert _key(pats) == (_key(po.mine_arrays(db.arrays(), minsup)[0]) if db is not single else []), i
    batch.close()


def test_the_static_workspace_ignores_the_limits():
    """Its levels hold two row sets and cannot wait for pieces."""
    db = gm.GraphDB.molecule(3, 100)
    db.upload()
    want = _key(gm.mine_noalloc(db, 20, collect_proj=True)[0])
    db.set_limits(piece_keys=500, list_units=1)
    assert _key(gm.mine_noalloc(db, 20, collect_proj=True)[0]) == want == _key(gm.mine(db, 20, collect_proj=True)[0])


def _bushy(n, seed=11):
    """Trees with a star of seven equal leaves each: many candidates a row."""
    rng = random.Random(seed)
    graphs = []
    for _ in range(n):
        labels, edges = tree(rng, 24, 3, 2, 3)
        k = len(labels)
        graphs.append((labels + [0] * 8, edges + [(k, k + i, 0) for i in range(1, 8)]))
    return graphs


LISTS = {
    "stars": ([star(n) for n in (1, 3, 9, 12, 12)], 1, 4, False),
    "cliques": ([clique(n) for n in (3, 5, 6, 9, 10)], 1, 3, False),
    "largest_star": ([star(63), star(40), clique(14)], 1, 2, False),
    "chosen_on_the_device": (_bushy(60), 6, 6, True),
}


@pytest.mark.parametrize("list_units", [1, 1200])  # no extent fits; a few do
@pytest.mark.parametrize("name", list(LISTS))
def test_lists_that_outgrow_their_pool(trace, name, list_units):
    graphs, minsup, max_edges, device = LISTS[name]
    db = gm.GraphDB.from_graphs(graphs)
    opats, ost = po.mine_arrays(db.arrays(), minsup, max_edges=max_edges)
    db.set_limits(list_units=list_units)
    for kw in ({}, {"canon_host": 2}, {"speculate": 2}):
        trace()
        pats, st = gm.mine(db, minsup, max_edges=max_edges, collect_proj=True, **kw)
        lines = trace().splitlines()
        again = [line for line in lines if int(re.search(r"lists_again (\d+)", line)[1]) > 0]
        assert again or (list_units > 1 and name == "stars")
        if device and "speculate" not in kw:
            assert any("device-chosen" in line for line in again)
        assert _key(pats) == _key(opats)
        assert (st["e_child"], st["e_cand"]) == (ost["e_child"], ost["e_cand"])
