"""GPU tests of the depth-first strategies against the CPU oracle at the limits of the wave's batches."""
import random

import pytest

import util
from test_gpu_maintenance import lib, random_edges, write_graph  # noqa: F401

pytestmark = pytest.mark.gpu

# n-cliques have n - 1 backward entries at the last depth (runs are kept for the first four); the path's
# frames fill and drain many times, the star's rows have one run each
QUERIES = {
    "clique6": (6, [(a, b) for b in range(6) for a in range(b)]),
    "path5": (5, [(a, a + 1) for a in range(4)]),
    "cycle6": (6, [(a, (a + 1) % 6) for a in range(6)]),
    "kite": (5, [(0, 1), (1, 2), (2, 0), (2, 3), (3, 4), (4, 0)]),
    "star": (5, [(0, k) for k in range(1, 5)]),
}


@pytest.mark.parametrize("batch", [3, 1200])  # fewer and more initial records than a depth-first search starts from
@pytest.mark.parametrize("strategy,local,product", [(0, True, True), (0, False, False), (1, True, False), (1, False, True)])
@pytest.mark.parametrize("directed", [False, True])
def test_depth_first_batches(lib, tmp_path, batch, strategy, local, product, directed):  # noqa: F811
    rng = random.Random(batch)
    n = 220
    labels = [rng.randrange(2) if v >= 6 else 0 for v in range(n)]
    edges = random_edges(rng, n, 2600, 1, directed, hub=6)
    rng.shuffle(edges)
    held, start = edges[:batch], edges[batch:]
    gone = start[:batch // 3]
    write_graph(tmp_path / "data.graph", labels, start)
    with open(tmp_path / "update.stream", "w") as f:
        f.write("".join(f"e {a} {b} {x}\n" for a, b, x in held) + "".join(f"-e {a} {b} {x}\n" for a, b, x in gone))
    paths = []
    for k, (nv, es) in enumerate(QUERIES.values()):
        write_graph(tmp_path / f"q{k}.graph", [rng.randrange(2) for _ in range(nv)], [(a, b, 0) for a, b in es], "t # 0\n")
        paths.append(str(tmp_path / f"q{k}.graph"))
    size = len(held) + len(gone)
    want, _ = util.oracle_stream(tmp_path / "data.graph", tmp_path / "update.stream", size, paths, threads=8, directed=directed)
    with lib.Session(device=0, directed=directed, ring_bytes=64 << 20, cp_list_bytes=32 << 20, lanes=4) as s:
        s.load_graph(str(tmp_path / "data.graph"))
        qids = [s.add_query(p) for p in paths]
        s.open_updates(str(tmp_path / "update.stream"), size)
        s.build()
        for q in qids:
            s.plan(q, lib.technique(matching_order=2, search_strategy=strategy, local_index=local, cartesian_product=product))
        for blocks in (64, 2048):
            s.set_tunables(dfs_blocks=blocks)
            s.snapshot()
            got = s.apply_batch(0)[0]
            s.restore()
            for k, name in enumerate(QUERIES):
                assert tuple(got[k]) == want[0, k], (name, blocks)
