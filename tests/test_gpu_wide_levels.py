"""BFS levels above the row limit (queries whose product suffix is counted in
batches): a level that fits at once, one written again at its size, one that
does not fit and is then not tried on the next batch, one without memory and
one past the deadline.

The graph has one layer of vertices per query vertex, so that the count is a
product of layer degrees: triangle 0-1-2 with a tail 2-3-4.  The new edges are
all pairs of layers 0 and 2 (90 000 seed rows); every pair of them has `fan`
common neighbours in layer 1, so the level has fan * 90 000 rows."""
import numpy as np
import pytest

from cgbdsm_amd import _native as N
from cgbdsm_amd.engine import CgbdsmError, Engine
from cgbdsm_amd.host import KeyBatch, Planner

pytestmark = pytest.mark.gpu

EDGES = [(0, 1), (0, 2), (1, 2), (2, 3), (3, 4)]
A = 300  # vertices of layers 0 and 2
ROWS = A * A


class Layers:
    """Keys of the layered graph: `index` (all but the edges 0-2) and `new`."""

    def __init__(self, fan, apart=0):
        """apart: neighbours in layer 1 that only one of the two layers has."""
        self.planner = Planner(np.arange(5, dtype=np.int32), np.array(EDGES, dtype=np.uint32))
        self.tables = self.planner.query_tables
        size = [A, fan + 2 * apart, A, 2 * A, 3]
        self.first = np.concatenate([[0], np.cumsum(size)])
        self.dv = int(self.first[-1])
        zero, two, one = np.arange(A), np.arange(A), np.arange(fan + apart)
        self.index = np.concatenate([
            self.keys(0, 1, np.repeat(zero, one.size), np.tile(one, A)),
            self.keys(2, 1, np.repeat(two, one.size), np.tile(one + apart, A)),
            self.keys(2, 3, np.repeat(two, 2), np.arange(2 * A)),  # two each
            self.keys(3, 4, np.repeat(np.arange(2 * A), 3), np.tile(np.arange(3), 2 * A))])  # three each
        self.new = self.keys(0, 2, np.repeat(zero, A), np.tile(two, A))
        self.count = ROWS * fan * 2 * 3

    def direction(self, a, b):
        return self.tables.eidx[a * N.MAX_QV + b]

    def keys(self, a, b, x, y):
        """Both directions of the edges x[i] of layer a - y[i] of layer b."""
        x, y = (x + self.first[a]).astype(np.uint64), (y + self.first[b]).astype(np.uint64)
        s = np.uint64(59)
        return np.concatenate([(np.uint64(self.direction(a, b)) << s) | (x << np.uint64(32)) | y,
                               (np.uint64(self.direction(b, a)) << s) | (y << np.uint64(32)) | x])

    def query(self, eng):
        q = eng.query(self.tables)
        q.index_init(self.index, self.dv)
        # The start edge is 0-2 (fewest entries), then vertex 1.
        card, avg = np.ones(q.ndir, dtype=np.uint32), np.ones(q.ndir, dtype=np.float32)
        card[self.direction(0, 2)] = card[self.direction(2, 0)] = 0
        plan = self.planner.make_plan(card, avg)
        assert [plan.go_vs[i] for i in range(5)] == [0, 2, 1, 3, 4]
        q.set_plan(plan)
        q.profile(True)
        return q

    def prepare(self, q, again=False):
        """The batch up to its matching (`again`: its edges leave first)."""
        none, ok = np.zeros(0, dtype=np.uint64), np.zeros(q.qe, dtype=np.uint8)
        ok[1] = 1  # only the query edge 0-2 has new edges
        q.stage(KeyBatch(0, none, self.new if again else none, self.new, ok, self.dv, 0, {}))
        q.transfer_update_all()
        assert q.transfer_update_index()
        q.build_local_index()
        q.kernel_times(reset=True)


def levels(q):
    """(level launches, depth and rows left for the DFS) of the last matching."""
    s = q.stats()
    return q.kernel_times()["extend"]["launches"], s["last_frontier_depth"], s["last_frontier_rows"]


@pytest.mark.parametrize("fan,want", [(3, (1, 3, 3 * ROWS)), (20, (2, 3, 20 * ROWS)), (100, (1, 2, ROWS))],
                         ids=["fits", "retried", "too-large"])
def test_wide_level(fan, want):
    print(f"case wide level {fan}", flush=True)
    eng, g = Engine(0), Layers(fan)
    q = g.query(eng)
    g.prepare(q)
    cnt, per = q.matching()
    assert cnt == g.count and per[1] == g.count
    assert levels(q) == want
    # The same batch again: the buffer has its size now, a level that did not fit is not tried.
    q.batch_update_global_index()
    g.prepare(q, again=True)
    assert q.matching()[0] == g.count
    assert levels(q) == ((1 if want[1] == 3 else 0),) + want[1:]
    q.close()
    eng.close()


def test_wide_level_without_memory():
    """The budget is what two batches take that count from the seeds."""
    print("case wide level memory", flush=True)
    g, need = Layers(20), 0
    for limit in (0, 65536):
        eng = Engine(0, need)
        q = g.query(eng)
        q.set_match_params(bfs_row_limit=limit)
        if need:
            assert np.array_equal(q.export(0), np.sort(g.index))  # its scratch is given back too
        for again in (False, True):
            g.prepare(q, again)
            assert q.matching()[0] == g.count
            assert levels(q)[1:] == (2, ROWS)
            q.batch_update_global_index()
        need = eng.memory()[0]
        q.close()
        eng.close()


def test_wide_level_past_the_deadline():
    """90 000 rows of 8 001 candidates each, one of them a common neighbour:
    several milliseconds, of which the kernel runs about two before it sees
    that the host asks it to stop."""
    print("case wide level deadline", flush=True)
    eng, g = Engine(0), Layers(1, apart=8000)
    q = g.query(eng)
    g.prepare(q)
    q.set_deadline(0.001)
    with pytest.raises(CgbdsmError) as ex:
        q.matching()
    assert ex.value.code == 5, ex.value  # CGBDSM_ERR_OVERFLOW
    asked = q.kernel_times()["extend"]["ms"]
    q.set_deadline(0)
    assert q.matching()[0] == g.count
    assert levels(q) == (1, 2, ROWS)  # the level was given up, the DFS counts from the seeds
    # Without a deadline a batch of the same size does not try it either; a new plan does.
    q.batch_update_global_index()
    g.prepare(q, again=True)
    assert q.matching()[0] == g.count
    assert levels(q) == (0, 2, ROWS)
    q.batch_update_global_index()
    q.set_plan(q.tables)
    g.prepare(q, again=True)
    assert q.matching()[0] == g.count
    whole = q.kernel_times()["extend"]["ms"]
    print(f"extend {asked} ms of {whole}", flush=True)
    assert levels(q) == (1, 3, ROWS)
    assert asked < whole
    q.close()
    eng.close()
