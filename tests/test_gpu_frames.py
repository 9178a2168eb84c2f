"""GPU tests of batches of partial results whose lists are long together: more candidates than one frame of
the depth-first search holds (2^24), and a sum past 32 bits.  The counts are closed forms, the hashes
are those of the breadth-first strategy, which has no frames."""
import numpy as np
import pytest

from test_gpu_maintenance import lib  # noqa: F401

pytestmark = pytest.mark.gpu


def write_lines(f, head, columns):
    """One line per row: `head` and the columns' decimal numbers, zero-padded."""
    columns = [np.asarray(c, dtype=np.int64) for c in columns]
    digits = [len(str(int(c.max()))) for c in columns]
    for a in range(0, len(columns[0]), 1 << 22):
        part = [c[a:a + (1 << 22)] for c in columns]
        line = [np.full(len(part[0]), ord(head), np.uint8)]
        for c, n in zip(part, digits):
            line.append(np.full(len(c), ord(" "), np.uint8))
            line += [(c // 10 ** d % 10 + ord("0")).astype(np.uint8) for d in reversed(range(n))]
        line.append(np.full(len(part[0]), ord("\n"), np.uint8))
        np.stack(line, 1).tofile(f)


def run(lib, tmp_path, labels, edges, held, query, techniques, **options):  # noqa: F811
    """Results of the one query for the batch of `held`, per technique, always from the same graph."""
    with open(tmp_path / "data.graph", "wb") as f:
        write_lines(f, "v", [np.arange(len(labels)), labels])
        write_lines(f, "e", [edges[0], edges[1], np.zeros(len(edges[0]))])
    with open(tmp_path / "update.stream", "wb") as f:
        write_lines(f, "e", [held[0], held[1], np.zeros(len(held[0]))])
    names, es = query
    (tmp_path / "q.graph").write_text("t # 0\n" + "".join(f"v {k} {x}\n" for k, x in enumerate(names)) + "".join(f"e {a} {b} 0\n" for a, b in es))
    got = []
    with lib.Session(device=0, **options) as s:
        s.load_graph(tmp_path / "data.graph")
        q = s.add_query(tmp_path / "q.graph")
        s.open_updates(tmp_path / "update.stream", len(held[0]))
        s.build()
        s.snapshot()
        for strategy, settings in techniques:
            print(f"case frames strategy={strategy} {settings}", flush=True)
            s.plan(q, lib.technique(search_strategy=strategy, cartesian_product=False))
            s.set_tunables(**settings)
            got.append(s.apply_batch(0)[0][0])
            s.restore()
    return got


def test_frame_sum_past_32_bits(lib, tmp_path):  # noqa: F811
    """64 partial results on one list of 2^26 keys: their lengths add up to 2^32.  The hub becomes a candidate only
    with the batch, so its steps are expected to be small and searched directly first."""
    middle, leaves = 64, 1 << 26
    labels = np.concatenate([[0, 1], np.full(middle, 2), np.full(leaves, 3)])
    ends = np.arange(2, len(labels))
    got = run(lib, tmp_path, labels, (np.zeros_like(ends), ends), ([0], [1]), ([0, 1, 2, 3], [(0, 1), (0, 2), (0, 3)]),
              [(3, {}), (2, {})], lanes=1)
    assert got[0][0] == middle * leaves
    assert got[1] == got[0]


@pytest.mark.parametrize("shape", ["rows_of_a_parent", "group_of_records"])
def test_frame_of_many_candidates_is_cut(lib, tmp_path, shape):  # noqa: F811
    """A few partial results of one batch share a long list, beside enough short ones that the depth-first kernel
    starts from these records: the frame takes only the rows that fit."""
    if shape == "rows_of_a_parent":  # hub 0: 64 vertices B, then 300,000 vertices C under each of them
        hubs, shared, long, b_of_hub = 4096, 1, 300_000, 64
        query = ([0, 1, 2, 3], [(0, 1), (0, 2), (0, 3)])
        want = b_of_hub * long + (hubs - 1)
    else:  # hub 0 is 64 records, and 64 records are a group
        hubs, shared, long, b_of_hub = 131_072, 64, 600_000, 0
        query = ([0, 1, 3, 4], [(0, 1), (0, 2), (2, 3)])
        want = shared * long + (hubs - 1)
    anchors = shared + hubs - 1
    A = hubs
    B = A + anchors
    b_n = b_of_hub + hubs - 1 if b_of_hub else 0
    C = B + b_n
    c_n = long + hubs - 1
    D = C + c_n  # every hub has an anchor vertex from the start, so that the summaries see its lists
    labels = np.concatenate([np.full(hubs, 0), np.full(anchors, 1), np.full(b_n, 2), np.full(c_n, 3), np.full(hubs, 1)])
    own = np.arange(1, hubs)
    src = [np.arange(hubs), np.zeros(long, dtype=np.int64), own]
    dst = [D + np.arange(hubs), C + np.arange(long), C + long + own - 1]
    if not b_n:  # every C has one neighbour below it
        labels = np.concatenate([labels, np.full(7, 4)])
        src.append(C + np.arange(c_n))
        dst.append(D + hubs + np.arange(c_n) % 7)
    else:
        src += [np.zeros(b_of_hub, dtype=np.int64), own]
        dst += [B + np.arange(b_of_hub), B + b_of_hub + own - 1]
    held = (np.concatenate([np.zeros(shared, dtype=np.int64), own]), A + np.arange(anchors))
    cases = [(3, {}), (1, {}), (1, {"dfs_blocks": 64}), (0, {"dfs_blocks": 64}), (0, {"dfs_blocks": 2048}), (2, {})]
    got = run(lib, tmp_path, labels, (np.concatenate(src), np.concatenate(dst)), held, query, cases, ring_bytes=1 << 30, cp_list_bytes=32 << 20, lanes=2)
    assert got[0][0] == want
    for k, g in enumerate(got):
        assert g == got[0], cases[k]
