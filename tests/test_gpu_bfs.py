"""GPU tests of the breadth-first strategy's device-side level chains against the CPU oracle: queries whose
levels end at the leaf, at a Cartesian-product tail of any length, or before the first level."""
import random

import pytest

import util
from test_gpu_maintenance import lib, random_edges, write_graph  # noqa: F401

pytestmark = pytest.mark.gpu

QUERIES = {
    "star": (5, [(0, k) for k in range(1, 5)]),
    "triangle_two_leaves": (5, [(0, 1), (1, 2), (2, 0), (0, 3), (1, 4)]),
    "triangle_one_leaf": (4, [(0, 1), (1, 2), (2, 0), (2, 3)]),
    "path4": (4, [(0, 1), (1, 2), (2, 3)]),
    "square": (4, [(0, 1), (1, 2), (2, 3), (3, 0)]),
    "clique5": (5, [(a, b) for b in range(5) for a in range(b)]),
}


@pytest.mark.parametrize("ring", [64 << 20, 4 << 20])  # the smaller one overflows: the host goes on with halves
@pytest.mark.parametrize("product", [True, False])
@pytest.mark.parametrize("team", [1, 4])  # a lane's own chain, a team's common one
def test_chained_breadth_first_levels(lib, tmp_path, monkeypatch, team, product, ring):  # noqa: F811
    monkeypatch.setenv("CSM_TEAM", str(team))
    rng = random.Random(5)
    n = 250
    labels = [rng.randrange(2) if v >= 5 else 0 for v in range(n)]
    edges = random_edges(rng, n, 2400, 1, False, hub=5)
    rng.shuffle(edges)
    held, start = edges[:500], edges[500:]
    gone = start[:150]
    write_graph(tmp_path / "data.graph", labels, start)
    with open(tmp_path / "update.stream", "w") as f:
        f.write("".join(f"e {a} {b} {x}\n" for a, b, x in held) + "".join(f"-e {a} {b} {x}\n" for a, b, x in gone))
    paths = []
    for k, (nv, es) in enumerate(QUERIES.values()):
        write_graph(tmp_path / f"q{k}.graph", [rng.randrange(2) for _ in range(nv)], [(a, b, 0) for a, b in es], "t # 0\n")
        paths.append(str(tmp_path / f"q{k}.graph"))
    size = len(held) + len(gone)
    want, _ = util.oracle_stream(tmp_path / "data.graph", tmp_path / "update.stream", size, paths, threads=8)
    with lib.Session(device=0, ring_bytes=ring, cp_list_bytes=32 << 20, lanes=8) as s:
        s.load_graph(str(tmp_path / "data.graph"))
        qids = [s.add_query(p) for p in paths]
        s.open_updates(str(tmp_path / "update.stream"), size)
        s.build()
        for q in qids:
            s.plan(q, lib.technique(matching_order=2, search_strategy=3, local_index=True, cartesian_product=product))
        got = s.apply_batch(0)[0]
        for k, name in enumerate(QUERIES):
            assert tuple(got[k]) == want[0, k], name
