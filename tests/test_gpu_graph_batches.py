"""Stream batches of the device graph at the sizes where their kernel changes
(up to 2048 pairs in one block, its keys sorted by one wavefront up to 64):
insertions and deletions mixed, repeated, already present or absent, self
loops and out-of-range ids.  The graph after the batch is compared through a
query attached to it and to a graph built from the expected edges."""
import numpy as np
import pytest

from cgbdsm_amd.engine import Engine
from cgbdsm_amd.host import Planner

pytestmark = pytest.mark.gpu


def _index(eng, graph, ql, qe):
    pl = Planner(ql, qe)
    q = eng.query(pl.query_tables)
    q.calig_attach(graph, ql)
    keys, ids = q.export(0), q.calig_old_ids()
    q.close()
    return keys, ids


@pytest.mark.parametrize("pairs", [1, 16, 32, 33, 512, 2047, 2048, 2049, 5000])
def test_graph_batch(pairs):
    print(f"case graph batch {pairs}", flush=True)
    rng = np.random.default_rng(pairs)
    n, m = 900, 12000
    labels = rng.integers(0, 2, n).astype(np.int32)

    def norm(e):
        e = e[(e[:, 0] != e[:, 1])]
        return {(min(a, b), max(a, b)) for a, b in e.tolist()}

    # a hub with several hundred neighbours beside random edges
    edges = np.concatenate([rng.integers(0, n, (m, 2)), np.stack([np.full(600, 5), rng.integers(0, n, 600)], 1)])
    before = norm(edges)
    present = np.array(sorted(before))
    half = max(1, pairs // 2)
    ins = rng.integers(0, n, (pairs - pairs // 2, 2))
    ins[: ins.shape[0] // 8] = present[rng.integers(0, len(present), ins.shape[0] // 8)]  # already there
    ins[-(ins.shape[0] // 8 + 1):] = ins[0]                                              # repeated (and pairs == 1)
    dele = present[rng.integers(0, len(present), pairs // 2)]
    dele[: dele.shape[0] // 8] = rng.integers(0, n, (dele.shape[0] // 8, 2))             # some absent
    stream = np.concatenate([ins, -dele - 1])
    rng.shuffle(stream)
    if pairs > 40:
        stream[3] = (n + 5, 2)
        stream[4] = (7, 7)
        stream[5] = (-3, 4)
    pos = stream[(stream >= 0).all(1) & (stream < n).all(1)]
    neg = -stream[(stream < 0).all(1)] - 1
    after = (before | norm(pos)) - ((norm(neg)) & before)
    assert half and len(after) > 0
    eng = Engine(0)
    g = eng.graph(labels, np.array(sorted(before)))
    g.set_stream(stream)
    g.apply_range(0, 2 * pairs)
    assert g.info()["directed_edges"] == 2 * len(after)
    want = eng.graph(labels, np.array(sorted(after)))
    ql, qe = np.array([0, 1, 0], dtype=np.int32), np.array([[0, 1], [1, 2]], dtype=np.uint32)
    for a, b in zip(_index(eng, g, ql, qe), _index(eng, want, ql, qe)):
        assert np.array_equal(a, b)
    g.close()
    want.close()
    eng.close()


@pytest.mark.parametrize("pairs", [16, 5000])
def test_closed_graph_gives_its_memory_back(pairs):
    print(f"case graph memory {pairs}", flush=True)
    rng = np.random.default_rng(pairs)
    eng = Engine(0)
    held = eng.memory()[0]
    g = eng.graph(rng.integers(0, 2, 900).astype(np.int32), rng.integers(0, 900, (4000, 2)))
    g.set_stream(rng.integers(0, 900, (pairs, 2)))
    g.apply_range(0, 2 * pairs)
    g.close()
    assert eng.memory()[0] == held
    eng.close()
