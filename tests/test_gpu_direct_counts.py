"""GPU tests that the direct steps' paths are taken (csm_get_direct_counts) while the results equal the CPU
oracle's: finished in the first pass, handed on, given up, beside the lanes' steps, more than one launch."""
import random

import pytest

import util
from test_gpu_direct import QUERIES
from test_gpu_maintenance import lib, random_edges, write_graph  # noqa: F401

pytestmark = pytest.mark.gpu


def run(lib, tmp_path, labels, start, held, gone, queries, strategies, **options):  # noqa: F811
    """Applies the batch, compares every query with the oracle and returns the counts.  queries: (vertex labels, edges)."""
    write_graph(tmp_path / "data.graph", labels, start)
    with open(tmp_path / "update.stream", "w") as f:
        f.write("".join(f"e {a} {b} {x}\n" for a, b, x in held) + "".join(f"-e {a} {b} {x}\n" for a, b, x in gone))
    paths = []
    for k, (names, es) in enumerate(queries):
        write_graph(tmp_path / f"q{k}.graph", names, [(a, b, 0) for a, b in es], "t # 0\n")
        paths.append(str(tmp_path / f"q{k}.graph"))
    size = len(held) + len(gone)
    want, _ = util.oracle_stream(tmp_path / "data.graph", tmp_path / "update.stream", size, paths, threads=8)
    with lib.Session(device=0, ring_bytes=64 << 20, cp_list_bytes=32 << 20, **options) as s:
        s.load_graph(str(tmp_path / "data.graph"))
        qids = [s.add_query(p) for p in paths]
        s.open_updates(str(tmp_path / "update.stream"), size)
        s.build()
        for k, q in enumerate(qids):
            s.plan(q, lib.technique(search_strategy=strategies[k % len(strategies)]))
        assert not any(s.direct_counts().values())
        got = s.apply_batch(0)[0]
        for k in range(len(queries)):
            assert tuple(got[k]) == want[0, k], queries[k]
        c = s.direct_counts()
    assert c["tried"] == c["finished"] + c["given_up"] + c["left_over"]
    return c


def small_graph(batch):
    rng = random.Random(batch)
    labels = [rng.randrange(3) if v >= 6 else 0 for v in range(300)]
    edges = random_edges(rng, 300, 3200, 1, False, hub=6)
    rng.shuffle(edges)
    held, start = edges[:batch], edges[batch:]
    return rng, labels, start, held, start[:batch // 3]


@pytest.mark.parametrize("direct", [1, 0])
@pytest.mark.parametrize("strategies", [(2,), (2, 3)])  # all steps may be direct; every second query's only
@pytest.mark.parametrize("batch", [3, 400])
def test_finished_first_or_beside_the_others(lib, tmp_path, monkeypatch, batch, strategies, direct):  # noqa: F811
    monkeypatch.setenv("CSM_DIRECT_STEPS", str(direct))
    monkeypatch.setenv("CSM_TEAM", "4")
    rng, labels, start, held, gone = small_graph(batch)
    names = QUERIES if len(strategies) > 1 else ("edge", "triangle", "clique6")  # no step of these is expected to be large
    queries = [([rng.randrange(3) for _ in range(QUERIES[k][0])], QUERIES[k][1]) for k in names]
    c = run(lib, tmp_path, labels, start, held, gone, queries, strategies, lanes=8)
    if not direct:
        assert not any(c.values())
        return
    assert c["finished"] > 0
    assert c["beside"] == (2 if len(strategies) > 1 else 0)


@pytest.mark.parametrize("beside", [False, True])
@pytest.mark.parametrize("leaves", [300, 1100])  # two free leaves: 90,000 candidates per update edge, 1,210,000 (more than a step may have)
def test_handed_on_and_given_up(lib, tmp_path, monkeypatch, leaves, beside):  # noqa: F811
    monkeypatch.setenv("CSM_TEAM", "2")
    rng = random.Random(leaves)
    labels = [0] + [1] * leaves + [2, 2, 2]
    hub = [(0, v, 0) for v in range(1, leaves + 4)]
    more = random_edges(rng, leaves, leaves, 1, False, hub=1)
    start = hub[:-2] + sorted({(a + 1, b + 1, x) for a, b, x in more})
    shapes = [(3, [(0, 1), (0, 2)]), (4, [(0, 1), (0, 2), (0, 3)]), (4, [(0, 1), (0, 2), (2, 3)]), (4, [(0, 1), (0, 2), (0, 3), (2, 3)])]
    queries = [([0, 2, 1, 1][:nv], es) for nv, es in shapes]
    strategies = [2] * len(queries)
    if beside:
        queries.append(queries[0])
        strategies.append(3)
    c = run(lib, tmp_path, labels, start, hub[-2:], start[:2], queries, strategies, lanes=4)
    assert c["handed_on"] > 0
    assert (c["given_up"] > 0) == (leaves == 1100)
    assert (c["beside"] > 0) == beside


def test_more_steps_than_one_launch_takes(lib, tmp_path):  # noqa: F811
    rng, labels, start, held, gone = small_graph(3)
    clique = [(a, b) for b in range(5) for a in range(b)]
    queries = [([rng.randrange(3) for _ in range(5)], clique) for _ in range(110)]
    c = run(lib, tmp_path, labels, start, held, gone, queries, (2,), lanes=64)
    assert c["tried"] == 2 * 110 * len(clique)  # both phases
    assert c["finished"] == c["tried"]


def test_a_step_that_fails_is_left_out_for_a_while(lib, tmp_path):  # noqa: F811
    """A step is expected to be small from the graph that the session was built on, where the hub has no vertex of
    label 2; the stream's every edge then has 1,100 squared candidates behind it."""
    leaves, batches = 1100, 12
    labels = [0] + [1] * leaves + [2] * batches
    write_graph(tmp_path / "data.graph", labels, [(0, v, 0) for v in range(1, leaves + 1)])
    (tmp_path / "update.stream").write_text("".join(f"e 0 {leaves + 1 + k} 0\n" for k in range(batches)))
    write_graph(tmp_path / "q.graph", [0, 2, 1, 1], [(0, 1, 0), (0, 2, 0), (0, 3, 0)], "t # 0\n")
    want, _ = util.oracle_stream(tmp_path / "data.graph", tmp_path / "update.stream", 1, [tmp_path / "q.graph"], threads=8)
    with lib.Session(device=0, ring_bytes=64 << 20, cp_list_bytes=32 << 20, lanes=4) as s:
        s.load_graph(str(tmp_path / "data.graph"))
        q = s.add_query(tmp_path / "q.graph")
        assert s.open_updates(str(tmp_path / "update.stream"), 1) == batches
        s.build()
        s.plan(q)
        s.snapshot()
        failed = []
        for _ in range(2):  # the restored session starts over
            for b in range(batches):
                assert tuple(s.apply_batch(b)[0][0]) == want[b, 0]
                c = s.direct_counts()
                failed.append(c["given_up"] + c["left_over"])
            s.restore()
    once = [1] * 9 + [2] * 3  # tried in the first phase, left out of eight, tried again
    assert failed == once + [2 + k for k in once]


@pytest.mark.parametrize("leaves", [20, 100])  # searched in one pass, handed on
def test_profile_sees_the_direct_search(lib, tmp_path, leaves):  # noqa: F811
    """Family 13 times the search passes and counts their algorithmic bytes (every row's list once, however often the
    row is handed on, and 4 per vertex found); a mask without it shows all steps in the other families."""
    labels = [0] + [1] * leaves + [2, 2]
    write_graph(tmp_path / "data.graph", labels, [(0, v, 0) for v in range(1, leaves + 2)])
    (tmp_path / "update.stream").write_text(f"e 0 {leaves + 2} 0\n")
    write_graph(tmp_path / "q.graph", [0, 2, 1, 1], [(0, 1, 0), (0, 2, 0), (0, 3, 0)], "t # 0\n")
    with lib.Session(device=0, ring_bytes=64 << 20, cp_list_bytes=32 << 20, lanes=4) as s:
        s.load_graph(str(tmp_path / "data.graph"))
        q = s.add_query(tmp_path / "q.graph")
        s.open_updates(str(tmp_path / "update.stream"), 1)
        s.build()
        s.plan(q)
        s.snapshot()
        got = {}
        for mask in (1 << 13, 1 << 8 | 1 << 9, 0):
            s.profile_enable(mask)
            tried = s.direct_counts()["tried"]
            got[mask] = s.apply_batch(0)[0][0], s.direct_counts()["tried"] - tried
            if mask:
                launches = {f: s.profile_read(f) for f in range(14)}
                if mask >> 13:
                    assert all((n > 0) == (f == 13) for f, (n, _, _) in launches.items())
                    assert launches[13][1] > 0
                    c = s.direct_counts()
                    assert c["finished"] == c["tried"] == 3 and (c["handed_on"] > 0) == (leaves == 100)
                    assert launches[13][2] == 4 * (leaves + leaves + leaves * leaves + leaves * (leaves - 1))
                else:
                    assert launches[13][0] == 0 and launches[8][0] + launches[9][0] > 0
            s.restore()
        assert got[1 << 13] == got[0] and got[0][1] == 3
        assert got[1 << 8 | 1 << 9] == (got[0][0], 0)
        assert got[0][0][0] == leaves * (leaves - 1)
