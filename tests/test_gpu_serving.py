"""Serving on the GPU: every request answered by the continuously batched
server (queries and mining jobs overlapping on the device) equals the same
request run alone -- exactly (integer supports and pattern sets)."""
import ctypes
import time

import pytest

import gpu_graph_mining_amd as gm
from gpu_graph_mining_amd import serving

pytestmark = pytest.mark.gpu


def test_served_results_equal_alone():
    db = gm.GraphDB.molecule(4, 1500)
    out = serving.serve(db, rate=2000.0, n_requests=48, seed=9, budget_bytes=1 << 30)
    reqs = out["_requests"]
    assert len(reqs) == 48 and all(r.done >= r.arrival for r in reqs)
    kinds = {r.kind for r in reqs}
    assert serving.QUERY in kinds and serving.MINING in kinds
    assert max(r.batch_size for r in reqs if r.kind == serving.QUERY) > 1  # batching happened
    for r in reqs:
        print("request", r.rid, r.kind, flush=True)
        assert r.result == serving.run_alone(db, r)
    assert out["query"]["p99_ms"] >= out["query"]["p50_ms"] > 0


def test_subset_batch_equals_each_subset_alone():
    """Jobs gathered on the device from the resident database (overlapping
    subsets, one empty) give each subset's own results."""
    db = gm.GraphDB.molecule(4, 3000)
    db.upload()
    subsets = [list(range(0, 3000, 3)), list(range(1, 2000, 2)), [5, 7, 11, 13, 2999], [], list(range(2500, 3000))]
    mins = [40, 60, 2, 1, 25]
    b = gm.Batch.from_subsets(db, subsets)
    try:
        res, _ = b.mine(mins, collect_proj=True)
    finally:
        b.close()
    for ids, m, got in zip(subsets, mins, res):
        if not ids:
            assert got == []
            continue
        sub = db.subset(ids)
        want, _ = gm.mine(sub, m, collect_proj=True)
        sub.close()
        assert sorted((tuple(c), s, n) for c, s, n in got) == sorted((tuple(c), s, n) for c, s, n in want)


@pytest.mark.parametrize("vlabels", [5, 90])  # the compact layout's alphabets, and beyond them
def test_subset_batches_take_over_buffers(vlabels):
    """Subset batches made one after the other from one database (larger,
    smaller, empty, duplicated graphs), two at a time, after a run that its
    sink stopped, and after more of them than are kept: each one's own
    results; a batch outlives its source."""
    db = gm.GraphDB.random(3, 400, 5, 9, 1.2, vlabels, 2)
    db.upload()

    def want(ids, minsup):
        sub = db.subset(ids)
        pats, st = gm.mine(sub, minsup, collect_proj=True)
        sub.close()
        return sorted((tuple(c), s, n) for c, s, n in pats), st["e_cand"]

    def check(batch, ids, minsup):
        res, st = batch.mine([minsup], collect_proj=True)
        got = sorted((tuple(c), s, n) for c, s, n in res[0])
        assert (got, st["e_cand"]) == (want(ids, minsup) if ids else ([], 0))

    jobs = [(list(range(40)), 6), (list(range(400)), 40), (list(range(0, 400, 7)), 6), ([], 1), ([9] * 12, 12),
            (list(range(399, 0, -2)), 20)]
    for ids, minsup in jobs + jobs[::-1]:
        print("alone", len(ids), flush=True)
        batch = gm.Batch.from_subsets(db, [ids])
        check(batch, ids, minsup)
        batch.close()
    live = [gm.Batch.from_subsets(db, [ids]) for ids, _ in jobs]
    for batch, (ids, minsup) in zip(live, jobs):
        print("among others", len(ids), flush=True)
        check(batch, ids, minsup)
    for batch in live:
        batch.close()
    lib = gm.load_library()
    batch = gm.Batch.from_subsets(db, [jobs[1][0]])
    stop = gm.JOB_PATTERN_CB(lambda *_: 1)
    assert lib.gm_batch_mine(batch._h, (gm.C.c_int32 * 1)(1), None, stop, None, None) != 0
    batch.close()
    wants = [want(*jobs[0]), want(*jobs[5])]
    last = [gm.Batch.from_subsets(db, [jobs[0][0]]), gm.Batch.from_subsets(db, [jobs[5][0]])]
    db.close()
    for batch, (_, minsup), w in zip(last, (jobs[0], jobs[5]), wants):
        res, st = batch.mine([minsup], collect_proj=True)
        assert (sorted((tuple(c), s, n) for c, s, n in res[0]), st["e_cand"]) == w
        batch.close()


def test_served_results_equal_alone_on_the_full_database():
    """The 50,000-graph molecule database: queries and mining jobs admitted
    into concurrent slots under a small memory budget (requests queue for
    memory), each result equal to the request run alone."""
    from gpu_graph_mining_amd import workloads as wl
    db = wl.config4()
    out = serving.serve(db, rate=1000.0, n_requests=40, seed=21, budget_bytes=256 << 20)
    reqs = out["_requests"]
    assert {r.kind for r in reqs} == {serving.QUERY, serving.MINING}
    for r in reqs:
        print("request", r.rid, r.kind, flush=True)
        assert r.result == serving.run_alone(db, r)
    assert out["bytes_per_unit"][serving.QUERY] > 0 and out["bytes_per_unit"][serving.MINING] > 0


@pytest.mark.parametrize("vlabels,minsups,least", [(5, [8, 4, 8], 20), (90, [2, 3, 2], 2)])  # compact and general kernels
def test_a_taken_over_batch_reports_its_own_memory(vlabels, minsups, least):
    """A small subset mined after a large one reports the peaks, call by call,
    that it has on a database that mined nothing before."""

    def fresh():
        db = gm.GraphDB.random(3, 400, 5, 9, 1.2, vlabels, 2)
        db.upload()
        return db

    def peaks(db, ids, minsups):
        batch = gm.Batch.from_subsets(db, [ids])
        got = [batch.mine([m])[1]["peak_device_bytes"] for m in minsups]
        batch.close()
        return got

    small, large = list(range(60)), list(range(400))
    want = peaks(fresh(), small, minsups)
    db = fresh()
    first = peaks(db, large, [least])
    assert first[0] > want[0]
    assert peaks(db, small, minsups) == want
    assert peaks(db, large, [least]) == first


@pytest.mark.parametrize("budget", [64 << 20, 8 << 30])
def test_kept_batches_stay_within_the_servers_budget(budget):
    """Mining requests of 10,000 molecules (some 220 MiB of buffers each): what
    the device holds when they are done is at most what the budget sets aside
    for the next ones (nothing of 64 MiB), and the handle's own limit is back
    after the server."""
    hip = gm.load_library()  # (the runtime that the library is linked with)
    db = gm.GraphDB.molecule(3, 30000)
    db.upload()

    def free():
        now, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(now), ctypes.byref(total)) == 0
        return now.value

    server = serving.Server(db, budget_bytes=budget, query_slots=1)
    before = free()
    requests = [serving.Request(serving.MINING, i, graphs=list(range(i, 30000, 3)), minsup=2000 - i, units=100000)
                for i in range(3)]
    for i, r in enumerate(requests):  # (one at a time: a batch of them holds more)
        server.submit(r)
        while len(server.finished) <= i and not server._errors:
            time.sleep(0.01)
    limit, reserve = serving.spare_bytes(budget, server.mining_slots)
    held = before - free()
    server.close()
    print("budget", budget, "held", held, "limit", limit, flush=True)
    assert held <= reserve and (held > 0) == (reserve > 0) and server.gate.budget + reserve == budget
    for r in requests:
        assert r.result == serving.run_alone(db, r)
    batch = gm.Batch.from_subsets(db, [requests[0].graphs])
    batch.mine([2000], count_only=True)
    used = before - free()
    batch.close()
    assert used > 100 << 20 and before - free() >= used  # kept: the default limit
    db.spare_limit(0)
    assert before - free() < used
    db.close()


@pytest.mark.parametrize("vlabels", [5, 90])  # two layouts on the device, and one
def test_the_server_knows_what_is_resident(vlabels):
    """What the estimates of a request's memory subtract from a run's peak is
    what the run finds on the device: a run that keeps no pattern has that
    peak, on the database and on a batch of its graphs."""
    db = gm.GraphDB.random(3, 400, 5, 9, 1.2, vlabels, 2)
    assert db.device_bytes() == 0
    server = serving.Server(db)
    resident = server.resident_bytes
    server.close()
    assert resident == db.device_bytes() == gm.mine(db, 401)[1]["peak_device_bytes"] > 0
    batch = gm.Batch.from_subsets(db, [list(range(100)), [7, 7]])
    assert batch.device_bytes() == batch.mine([101, 3])[1]["peak_device_bytes"] > 0
    batch.close()


def test_subsets_past_32_bit_offsets_are_refused():
    """One graph selected so often that the gathered adjacency (65,280 entries
    a time) passes 2^31: refused before anything is gathered."""
    n = 256
    db = gm.GraphDB.from_graphs([([0] * n, [(a, b, 0) for a in range(n) for b in range(a + 1, n)])])
    with pytest.raises(gm.GMError) as e:
        gm.Batch.from_subsets(db, [[0] * 33000])
    assert e.value.code == gm.GM_E_UNSUPPORTED
    batch = gm.Batch.from_subsets(db, [[0] * 3])
    assert batch.mine([4])[0] == [[]]
    batch.close()
