"""GPU tests of the direct steps (small steps searched from their anchors in one launch, rest handed on
pass by pass) against the CPU oracle, and of the steps beside them with direct steps switched off."""
import random

import pytest

import util
from test_gpu_maintenance import lib, random_edges, write_graph  # noqa: F401

pytestmark = pytest.mark.gpu

# one edge (no vertex to search), n-cliques of more backward entries than are kept per row, paths and trees
# whose frames fill and drain many times, a seven-vertex cycle
QUERIES = {
    "edge": (2, [(0, 1)]),
    "triangle": (3, [(0, 1), (1, 2), (2, 0)]),
    "clique6": (6, [(a, b) for b in range(6) for a in range(b)]),
    "path5": (5, [(a, a + 1) for a in range(4)]),
    "cycle7": (7, [(a, (a + 1) % 7) for a in range(7)]),
    "kite": (5, [(0, 1), (1, 2), (2, 0), (2, 3), (3, 4), (4, 0)]),
    "star": (5, [(0, k) for k in range(1, 5)]),
}


def check(lib, tmp_path, labels, start, held, gone, queries, query_labels, directed, lanes):  # noqa: F811
    write_graph(tmp_path / "data.graph", labels, start)
    with open(tmp_path / "update.stream", "w") as f:
        f.write("".join(f"e {a} {b} {x}\n" for a, b, x in held) + "".join(f"-e {a} {b} {x}\n" for a, b, x in gone))
    paths = []
    for k, (nv, es) in enumerate(queries.values()):
        write_graph(tmp_path / f"q{k}.graph", [query_labels(k, v) for v in range(nv)], [(a, b, 0) for a, b in es], "t # 0\n")
        paths.append(str(tmp_path / f"q{k}.graph"))
    size = len(held) + len(gone)
    want, _ = util.oracle_stream(tmp_path / "data.graph", tmp_path / "update.stream", size, paths, threads=8, directed=directed)
    with lib.Session(device=0, directed=directed, ring_bytes=64 << 20, cp_list_bytes=32 << 20, lanes=lanes) as s:
        s.load_graph(str(tmp_path / "data.graph"))
        qids = [s.add_query(p) for p in paths]
        s.open_updates(str(tmp_path / "update.stream"), size)
        s.build()
        for q in qids:
            s.plan(q)
        s.snapshot()
        for depth in (16, 2):  # a stack depth that leaves the deeper queries to the other path
            s.set_tunables(stack_depth=depth)
            got = s.apply_batch(0)[0]
            s.restore()
            for k, name in enumerate(queries):
                assert tuple(got[k]) == want[0, k], (name, depth)


@pytest.mark.parametrize("direct", [1, 0])
@pytest.mark.parametrize("lanes", [4, 64])  # more steps than lanes: tried beside the others; fewer: first
@pytest.mark.parametrize("batch", [3, 400])
@pytest.mark.parametrize("directed", [False, True])
def test_direct_steps(lib, tmp_path, monkeypatch, direct, lanes, batch, directed):  # noqa: F811
    monkeypatch.setenv("CSM_DIRECT_STEPS", str(direct))
    rng = random.Random(batch)
    n = 300
    labels = [rng.randrange(3) if v >= 6 else 0 for v in range(n)]
    edges = random_edges(rng, n, 3200, 1, directed, hub=6)
    rng.shuffle(edges)
    held, start = edges[:batch], edges[batch:]
    check(lib, tmp_path, labels, start, held, start[:batch // 3], QUERIES, lambda k, v: 0 if k in (1, 2) else rng.randrange(3), directed, lanes)


@pytest.mark.parametrize("leaves", [127, 513, 1100])  # under a round, just over a piece, several pieces and passes
def test_rest_of_a_hub_is_handed_on(lib, tmp_path, leaves):  # noqa: F811
    """Few anchors with long lists behind them: rows are cut into pieces and searched by later passes, up to
    more candidates than a step may have (two free leaves of a hub: 1,100 squared)."""
    rng = random.Random(leaves)
    labels = [0] + [1] * leaves + [2, 2, 2]
    hub = [(0, v, 0) for v in range(1, leaves + 4)]
    more = random_edges(rng, leaves, leaves, 1, False, hub=1)
    start = hub[:-2] + sorted({(a + 1, b + 1, x) for a, b, x in more})
    held, gone = hub[-2:], start[:2]
    queries = {
        "one_leaf": (3, [(0, 1), (0, 2)]),
        "two_leaves": (4, [(0, 1), (0, 2), (0, 3)]),
        "hop": (4, [(0, 1), (0, 2), (2, 3)]),
        "closed": (4, [(0, 1), (0, 2), (0, 3), (2, 3)]),
    }
    check(lib, tmp_path, labels, start, held, gone, queries, lambda k, v: [0, 2, 1, 1][v], False, 4)
