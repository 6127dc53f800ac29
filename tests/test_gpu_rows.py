"""Index records when the vertex count outgrows their row stride: M, the update
index and its touched rows move with it, in both layouts.  Expected keys by
numpy set operations."""
import numpy as np
import pytest

from cgbdsm_amd.engine import Engine
from cgbdsm_amd.host import KeyBatch, Planner

pytestmark = pytest.mark.gpu

USHIFT = 59  # ebits 5


def _keys(rng, n, dv):
    d = rng.integers(0, 4, n).astype(np.uint64)
    u, v = (rng.integers(0, dv, n).astype(np.uint64) for _ in range(2))
    return (d << np.uint64(USHIFT)) | (u << np.uint64(32)) | v


@pytest.mark.parametrize("layout", ["gamma", "gpma"])
@pytest.mark.parametrize("sizes", [(1, 1024, 1025, 1026), (700, 1536, 1537, 9000), (3000, 3001, 4500, 4501, 7000)])
def test_vertices_outgrow_the_stride(layout, sizes):
    print(f"case rows {layout} {sizes}", flush=True)
    rng = np.random.default_rng(sum(sizes))
    pl = Planner(np.array([0, 1, 2], dtype=np.int32), np.array([[0, 1], [1, 2]], dtype=np.uint32))
    eng = Engine(0)
    q = eng.query(pl.query_tables)
    q.set_layout(layout)
    want = np.unique(_keys(rng, 5000, sizes[0]))
    card, avg = q.index_init(want, sizes[0])
    q.set_plan(pl.make_plan(card, avg))
    upd = np.zeros(0, dtype=np.uint64)
    for dv in sizes:
        # (the last owner and target of each size among the keys)
        last = np.uint64(dv - 1)
        ins = np.concatenate([_keys(rng, 3000, dv), [(np.uint64(3) << np.uint64(USHIFT)) | (last << np.uint64(32)) | last]])
        dele = want[:: 7]
        new = np.unique(_keys(rng, 500, dv))
        q.stage(KeyBatch(0, ins, dele, new, np.ones(q.qe, dtype=np.uint8), dv, 0, {}))
        assert np.array_equal(np.sort(q.export(1)), upd)  # the last batch's, on moved rows
        q.transfer_update_all()
        want = np.setdiff1d(np.union1d(want, ins), dele)
        assert np.array_equal(q.export(0), want)
        q.transfer_update_index()
        upd = new
        assert np.array_equal(np.sort(q.export(1)), upd)
        q.batch_update_global_index()
        want = np.union1d(want, upd)
    q.close()
    eng.close()
