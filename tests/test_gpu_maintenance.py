"""GPU tests of the batch maintenance kernels against plain Python over the updated edge set."""
import random
from collections import Counter

import numpy as np
import pytest

import util

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    util.ensure_built()
    return util.ffi()


def write_graph(path, labels, edges, head=""):
    with open(path, "w") as f:
        f.write(head + "".join(f"v {v} {x}\n" for v, x in enumerate(labels)))
        f.write("".join(f"e {a} {b} {x}\n" for a, b, x in edges))


def random_edges(rng, n, m, elabels, directed, hub=0):
    """m distinct edges over n vertices; the first `hub` vertices take part in half of them."""
    seen = {}
    while len(seen) < m:
        a, b = rng.randrange(hub) if hub and rng.random() < 0.5 else rng.randrange(n), rng.randrange(n)
        if a == b or (a, b) in seen or (not directed and (b, a) in seen):
            continue
        seen[a, b] = rng.randrange(elabels)
    return [(a, b, x) for (a, b), x in seen.items()]


def groups_of(nv, edges, labels, directed):
    """Per vertex: number of neighbours by (direction, edge label, neighbour label)."""
    got = [Counter() for _ in range(nv)]
    for a, b, x in edges:
        got[a][0, x, labels[b]] += 1
        got[b][1 if directed else 0, x, labels[a]] += 1
    return got


# a star's centre has one group per leaf label: fewer, as many and more than the run lookups the
# candidate kernel issues together (4)
@pytest.mark.parametrize("leaves,directed,batch", [(1, False, 1), (4, False, 63), (5, False, 257), (9, False, 700), (4, True, 65), (6, True, 400)])
def test_candidates_after_batches(lib, tmp_path, leaves, directed, batch):
    rng = random.Random(leaves * 1000 + batch)
    n, nl, el = 300, 5, 2
    labels = [rng.randrange(nl) for _ in range(n)]
    edges = random_edges(rng, n, 2600, el, directed)
    rng.shuffle(edges)
    held, start = edges[:batch], edges[batch:]
    gone = start[:batch // 2]
    write_graph(tmp_path / "data.graph", labels, start)
    # label nl has no query vertex; one query holds a label the data graph lacks
    star = [rng.randrange(nl - 1) for _ in range(leaves + 1)]
    queries = [(star, [(0, k, rng.randrange(el)) if k % 2 or not directed else (k, 0, rng.randrange(el)) for k in range(1, leaves + 1)]),
               ([0, 1, 2], [(0, 1, 0), (1, 2, 1)]), ([0, nl + 3], [(0, 1, 0)])]
    with open(tmp_path / "update.stream", "w") as f:
        f.write("".join(f"e {a} {b} {x}\n" for a, b, x in held) + "".join(f"-e {a} {b} {x}\n" for a, b, x in gone))
    with lib.Session(device=0, directed=directed, ring_bytes=64 << 20, cp_list_bytes=32 << 20) as s:
        s.load_graph(str(tmp_path / "data.graph"))
        ids = []
        for k, (labs, es) in enumerate(queries):
            write_graph(tmp_path / f"q{k}.graph", labs, es, "t # 0\n")
            ids.append(s.add_query(str(tmp_path / f"q{k}.graph")))
        nb = s.open_updates(str(tmp_path / "update.stream"), len(held) + len(gone))
        s.build()
        for q in ids:
            s.plan(q)
        for b in range(nb):
            s.apply_batch(b)
        now = groups_of(n, [e for e in start if e not in set(gone)] + held, labels, directed)
        for q, (labs, es) in zip(ids, queries):
            need = groups_of(len(labs), es, labs, directed)
            for u, x in enumerate(labs):
                want = [v for v in range(n) if labels[v] == x and all(now[v][k] >= c for k, c in need[u].items())]
                words = s.candidates(q, u)
                assert [v for v in range(n) if words[v >> 5] >> (v & 31) & 1] == want, (q, u)


def run_batch(s, edges, gone):
    rows = np.array([(a, b, 0) for a, b in edges], dtype=np.uint32).reshape(-1, 3)
    return s.apply_edges(np.ascontiguousarray(rows[:, 0]), np.ascontiguousarray(rows[:, 1]), np.ascontiguousarray(rows[:, 2]),
                         np.array(gone, dtype=np.uint8))[0]


# delta segments around the limits of a lane's registers (8), a wave (64), a wave's LDS slice (512) and
# a block's LDS (8192), with the other segments of the batch short
@pytest.mark.parametrize("arcs", [1, 8, 9, 64, 65, 512, 513, 8192, 8193])
@pytest.mark.parametrize("directed", [False, True])
def test_delta_segments(lib, tmp_path, arcs, directed):
    rng = random.Random(arcs)
    n = arcs + 400
    hub = rng.randrange(n)
    spokes = rng.sample([v for v in range(n) if v != hub], arcs)
    ring = [(v, (v + 1) % n) for v in range(0, n - 1, 2) if hub not in (v, v + 1)]  # one arc per vertex, deleted and put back
    star = [(hub, v) if rng.random() < 0.5 else (v, hub) for v in spokes]
    write_graph(tmp_path / "data.graph", [0] * n, [(a, b, 0) for a, b in ring])
    write_graph(tmp_path / "q.graph", [0, 0], [(0, 1, 0)], "t # 0\n")
    with lib.Session(device=0, directed=directed, max_batch_edges=2 * n, ring_bytes=64 << 20, cp_list_bytes=32 << 20) as s:
        s.load_graph(str(tmp_path / "data.graph"))
        q = s.add_query(str(tmp_path / "q.graph"))
        s.build()
        s.plan(q)

        def lists(edges):
            out, inn = [[] for _ in range(n)], [[] for _ in range(n)]
            for a, b in edges:
                out[a].append(b)
                (inn if directed else out)[b].append(a)
            return [sorted(x) for x in out], [sorted(x) for x in inn]

        def check(edges):
            out, inn = lists(edges)
            for v in [hub] + rng.sample(range(n), 60):
                assert list(s.adjacency(v)) == out[v], v
                if directed:
                    assert list(s.adjacency(v, 1)) == inn[v], v

        twice = star + [star[-1]]  # the same arc twice, in the hub's segment
        for bad in (twice, twice if directed else star + [star[0][::-1]], star + [ring[0]]):
            with pytest.raises(lib.CsmError):
                run_batch(s, bad, [0] * len(bad))
        with pytest.raises(lib.CsmError):
            run_batch(s, star, [1] * len(star))
        check(ring)
        both = star + ring
        rng.shuffle(both)
        fresh = set(star)
        # the query is one edge: its embeddings are the anchors, the hub's all in one run
        way = 1 if directed else 2
        got = run_batch(s, both, [0 if e in fresh else 1 for e in both])
        assert tuple(got[0])[:2] == (way * len(star), way * len(ring))
        check(star)
        got = run_batch(s, both, [1 if e in fresh else 0 for e in both])
        assert tuple(got[0])[:2] == (way * len(ring), way * len(star))
        check(ring)
