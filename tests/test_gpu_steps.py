"""Batched product-suffix steps over long lists: a step that reaches its entry
budget ends early and goes on at the next sibling, whose candidate range other
wavefronts may take over at any candidate.  Counts against the oracle, from
the depth-2 seeds and from the rows of the BFS levels; the number of steps
where it follows from the lists' lengths."""
import numpy as np
import pytest

from cgbdsm_amd import _native as N
from cgbdsm_amd.engine import Engine
from cgbdsm_amd.host import HostSession, KeyBatch, Planner, synth_spec
from tests import parity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("params", [{"bfs_row_limit": 0}, {"bfs_row_limit": 65536},
                                    {"bfs_row_limit": 0, "donate_min": 1}],
                         ids=["seeds", "rows", "split"])
@pytest.mark.parametrize("case", [(10, 60, 2, 4, "dense", 3), (9, 90, 1, 4, "dense", 5), (10, 40, 3, 5, "dense", 3),
                                  (9, 60, 2, 5, "tree", 6)],
                         ids=["l2-dense4", "l1-dense4", "l3-dense5", "l2-tree5"])
def test_long_steps(eng, case, params):
    scale, deg, labels, qs, kind, seed = case
    print(f"case steps {case} {params}", flush=True)
    spec = synth_spec(scale, deg, labels, seed=seed, query_size=qs, query_kind=kind, query_seed=seed)
    host = HostSession(spec=spec, batch_edges=200, threads=4)
    res = parity.run_stream(host, eng, check_index=False, check_masks=False, max_batches=2, match_params=params)
    print(f"total {res['total']}, batched suffix steps {res['dfs_batched']}", flush=True)
    assert res["batches"] > 0
    assert res["mismatches"] == 0
    # (the tree's suffix has two positions of one label: counted sibling by sibling)
    assert (res["dfs_batched"] > 0) == (kind == "dense")


@pytest.mark.parametrize("length,steps", [(32, 1), (33, 2), (100, 4), (3000, 64)])
def test_steps_end_at_the_budget(eng, length, steps):
    """One new edge 0-1 of a 4-clique, 64 siblings at position 2 with lists of
    `length` entries each at position 3: a step ends before the first sibling
    past the budget of 2048 entries, but always counts its first one."""
    print(f"case step budget {length}", flush=True)
    edges = [(0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3)]
    pl = Planner(np.arange(4, dtype=np.int32), np.array(edges, dtype=np.uint32))
    t = pl.query_tables
    size = [1, 1, 64, length]
    first = np.concatenate([[0], np.cumsum(size)])

    def keys(a, b):  # every pair of the two layers, both directions
        x = np.repeat(np.arange(size[a]) + first[a], size[b]).astype(np.uint64)
        y = np.tile(np.arange(size[b]) + first[b], size[a]).astype(np.uint64)
        return np.concatenate([(np.uint64(t.eidx[c * N.MAX_QV + d]) << np.uint64(59)) | (u << np.uint64(32)) | v
                               for c, d, u, v in ((a, b, x, y), (b, a, y, x))])

    q = eng.query(t)
    q.index_init(np.concatenate([keys(a, b) for a, b in edges[1:]]), int(first[-1]))
    card = np.ones(q.ndir, dtype=np.uint32)
    card[t.eidx[1]] = card[t.eidx[N.MAX_QV]] = 0  # the start edge is 0-1
    plan = pl.make_plan(card, np.ones(q.ndir, dtype=np.float32))
    assert [plan.go_vs[i] for i in range(4)] == [0, 1, 2, 3]
    q.set_plan(plan)
    q.set_match_params(donate_min=0)
    none, ok = np.zeros(0, dtype=np.uint64), np.zeros(q.qe, dtype=np.uint8)
    ok[0] = 1
    q.stage(KeyBatch(0, none, none, keys(0, 1), ok, int(first[-1]), 0, {}))
    assert q.run_batch()[0] == 64 * length
    assert q.stats()["last_dfs_batched"] == steps
    q.close()
