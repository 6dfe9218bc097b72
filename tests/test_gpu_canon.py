"""The minimum-DFS-code check on the device (csrc/canon.hip, one wave per
code) against the host check (csrc/canonical.cpp) and the oracle's
restatement of ismin.cpp (src/gspan/ismin.cpp:36-140), alone through
gm_dfs_codes_are_min and inside mining, where it decides every level's
frequent keys before their download."""
import random

import pytest

import gpu_graph_mining_amd as gm
from oracle import py_oracle as po

from helpers import case_db, check_listing, listing
from test_host import _rand_code
from test_oracle import ISMIN_KAT

pytestmark = pytest.mark.gpu


def _big_code(rng, n):
    """A random DFS traversal of a random connected labelled graph of n
    vertices with extra edges (as test_host._rand_code, larger)."""
    labels = [rng.randint(0, 3) for _ in range(n)]
    edges = {(rng.randrange(v), v) for v in range(1, n)}
    for _ in range(rng.randint(0, n)):
        a, b = rng.sample(range(n), 2)
        edges.add((min(a, b), max(a, b)))
    el = {e: rng.randint(0, 2) for e in edges}
    adj = {v: [] for v in range(n)}
    for a, b in edges:
        adj[a].append(b)
        adj[b].append(a)
    order, code, used = {0: 0}, [], set()

    # DFS with the backward edges of each vertex first, as gSpan lists them
    # (smallest discovery index first)
    def visit(u):
        for w in sorted((w for w in adj[u] if w in order and (min(u, w), max(u, w)) not in used),
                        key=lambda w: order[w]):
            used.add((min(u, w), max(u, w)))
            code.append((order[u], order[w], labels[u], el[(min(u, w), max(u, w))], labels[w]))
        nb = adj[u][:]
        rng.shuffle(nb)
        for w in nb:
            if w not in order:
                order[w] = len(order)
                used.add((min(u, w), max(u, w)))
                code.append((order[u], order[w], labels[u], el[(min(u, w), max(u, w))], labels[w]))
                visit(w)

    visit(0)
    return code


def test_device_check_matches_host_and_oracle_on_random_codes():
    rng = random.Random(11)
    codes = [_rand_code(rng) for _ in range(4000)]
    got = gm.codes_are_min(codes)
    n_min = 0
    for c, g in zip(codes, got):
        want = po.is_min(po.normalize(c))
        assert g == want, c
        n_min += want
    assert 300 < n_min < 3700


def test_device_check_on_larger_codes():
    """Codes of 8-30 vertices (up to 60 edges): the same answers as the
    host check and the oracle."""
    rng = random.Random(12)
    codes = [_big_code(rng, rng.randint(8, 30)) for _ in range(600)]
    codes = [c for c in codes if len(c) <= 64]
    got = gm.codes_are_min(codes)
    for c, g in zip(codes, got):
        assert g == gm.DFSCode(c).is_min() == po.is_min(po.normalize(c)), c


def test_device_check_known_answers_and_wildcards():
    codes = [gm.DFSCode.read_from_str(s) for s, _ in ISMIN_KAT]
    assert gm.codes_are_min(codes) == [e for _, e in ISMIN_KAT]
    rng = random.Random(13)
    full = [_rand_code(rng) for _ in range(500)]
    wild = [gm.DFSCode(c).wildcard() for c in full]
    assert gm.codes_are_min(wild) == [gm.DFSCode(c).is_min() for c in wild]


def test_device_check_symmetric_codes_beyond_its_capacity():
    """Stars with identical leaves: a prefix of k leaves has 9!/(9-k)!
    embeddings in a 9-leaf star, beyond the device's 64 from two leaves
    on; such codes are checked on the host with the same answers."""
    star = [(0, i, 0, 0, 1) for i in range(1, 10)]
    # the same star entered from a leaf: the grown code leaves the centre
    # first, so the second tuple differs
    bad = [(0, 1, 1, 0, 0)] + [(1, i, 0, 0, 1) for i in range(2, 10)]
    got = gm.codes_are_min([star, bad])
    assert got == [gm.DFSCode(star).is_min(), gm.DFSCode(bad).is_min()]
    assert got == [True, False]


def test_device_check_rejects_malformed_codes():
    with pytest.raises(gm.GMError):
        gm.codes_are_min([[(0, 0, 1, 0, 1)]])


@pytest.mark.parametrize("name", ["chem_34", "chem_10", "config1_1k", "config4_2k", "labeled_2",
                                  "get_labeled_test_database_2"])
def test_mining_device_and_host_checks_agree(golden, name):
    """The same patterns, supports and |Proj| whichever side checks (the
    device on every level, the host on every level, the adaptive default),
    and the reference's listing (the device leaves a few highly symmetric
    codes of the molecule databases to the host)."""
    case = golden[name]
    db = case_db(case)
    dev, sd = gm.mine(db, case["minsup"], collect_proj=True, canon_host=2)
    host, sh = gm.mine(db, case["minsup"], collect_proj=True, canon_host=1)
    auto, sa = gm.mine(db, case["minsup"], collect_proj=True)
    check_listing(listing(dev), case)
    key = lambda pats: sorted((tuple(c), s, n) for c, s, n in pats)
    assert key(dev) == key(host) == key(auto)
    for k in ("n_patterns", "e_child", "e_root", "e_cand"):
        assert sd[k] == sh[k] == sa[k], k
    assert sh["canon_host_keys"] == 0 and sd["canon_host_keys"] <= sd["n_candidates"] // 100


def test_mining_with_keys_left_to_the_host():
    """Five 9-leaf stars (centre label 0, leaves 1): every star pattern of
    two or more leaves is beyond the device check's capacity and goes to
    the host; the result equals the oracle's."""
    n, leaves = 5, 9
    vb, vl, eb, ef, et, el = [0], [], [0], [], [], []
    for _ in range(n):
        vl += [0] + [1] * leaves
        vb.append(len(vl))
        ef += [0] * leaves
        et += list(range(1, leaves + 1))
        el += [0] * leaves
        eb.append(len(ef))
    db = gm.GraphDB.from_arrays(vb, vl, eb, ef, et, el)
    pats, st = gm.mine(db, n, collect_proj=True, canon_host=2)
    assert st["canon_host_keys"] > 0
    opats, ost = po.mine_arrays(db.arrays(), n)
    assert sorted((po.normalize(c), s, p) for c, s, p in pats) == sorted((c, s, p) for c, s, p in opats)
    assert st["e_child"] == ost["e_child"] and st["n_patterns"] == leaves


@pytest.mark.parametrize("n", [31, 32, 33, 36])
def test_device_check_with_many_images_of_the_root(n):
    """A path of n equal edges: its root tuple has 2 n images, up to and past
    the 64 embeddings the device holds (more are left to the host)."""
    path = [(i, i + 1, 0, 0, 0) for i in range(n)]
    # the same path grown from its second vertex: not minimal
    other = [(0, 1, 0, 0, 0)] + [(i, i + 1, 0, 0, 0) for i in range(1, n - 1)] + [(0, n, 0, 0, 0)]
    want = [gm.DFSCode(c).is_min() for c in (path, other)]
    assert want == [True, False]
    assert gm.codes_are_min([path, other]) == want
