"""A memory budget that cuts the root level: the 1-edge patterns are then
mined group by group, so no group's 2-edge patterns are all of the
database's, and the 2-edge path rule must not take them for that.  Whatever
the budget, the patterns and their counts are the oracle's."""
import random

import pytest

import gpu_graph_mining_amd as gm
from oracle import py_oracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("labels", [5, 9])  # both layouts of the level rows
def test_budgets_that_cut_the_root_level(labels):
    rng = random.Random(85 + labels)
    graphs = []
    for _ in range(40):
        graphs.append(([rng.randrange(5) for _ in range(20)] + list(range(labels)),
                       [(rng.randrange(v), v, rng.randrange(labels)) for v in range(1, 20 + labels)]))
    db = gm.GraphDB.from_graphs(graphs)
    opats, ost = po.mine_arrays(db.arrays(), 2, max_edges=4)
    want = {po.normalize(c): (s, n) for c, s, n in opats}
    for budget in (2000, 6000, 12000, 20000, 40000, 80000):
        print("labels", labels, "budget", budget, flush=True)
        pats, st = gm.mine(db, 2, max_edges=4, collect_proj=True, mem_budget=budget)
        assert {po.normalize(c): (s, n) for c, s, n in pats} == want
        assert (st["e_child"], st["e_cand"]) == (ost["e_child"], ost["e_cand"])
