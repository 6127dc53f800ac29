"""Index maintenance of single lists at the lengths where its kernels change:
one lane, one wavefront, a whole block (lists of 4096 entries or more, moved
4096 entries per step).  Expected lists by numpy set operations."""
import numpy as np
import pytest

from cgbdsm_amd.engine import Engine
from cgbdsm_amd.host import KeyBatch, Planner

pytestmark = pytest.mark.gpu

USHIFT = 59  # ebits 5


def _key(d, u, v):
    return (np.uint64(d) << np.uint64(USHIFT)) | (np.uint64(u) << np.uint64(32)) | np.asarray(v, dtype=np.uint64)


def _batch(ins, dele, dv, qe):
    none = np.zeros(0, dtype=np.uint64)
    return KeyBatch(0, ins, dele, none, np.zeros(qe, dtype=np.uint8), dv, 0, {})


@pytest.mark.parametrize("n", [1, 47, 300, 4095, 4096, 4097, 8192, 12289, 40000])
@pytest.mark.parametrize("k", [1, 63, 64, 1500])
def test_one_list_insert_then_remove(n, k):
    print(f"case list n={n} k={k}", flush=True)
    rng = np.random.default_rng(n * 131 + k)
    dv = 4 * (n + k) + 1000
    pl = Planner(np.array([0, 1, 2], dtype=np.int32), np.array([[0, 1], [1, 2]], dtype=np.uint32))
    eng = Engine(0)
    q = eng.query(pl.query_tables)
    pool = rng.permutation(dv - 500)[: n + 2 * k].astype(np.uint64)
    held = _key(1, 7, pool[:n])
    small = _key(0, 9, np.arange(5))  # a neighbouring short list stays as it is
    card, avg = q.index_init(np.concatenate([held, small]), dv)
    q.set_plan(pl.make_plan(card, avg))
    want = np.sort(np.concatenate([held, small]))
    # new values in two steps (the list grows its extent, then fits its slack),
    # half of the batch present already and some of it twice
    for part in (pool[n: n + k], pool[n + k:]):
        ins = np.concatenate([_key(1, 7, part), held[: min(n, k)], _key(1, 7, part[:3])])
        q.stage(_batch(ins, np.zeros(0, dtype=np.uint64), dv, q.qe))
        q.transfer_update_all()
        q.transfer_update_index()
        want = np.union1d(want, ins)
        assert np.array_equal(q.export(0), want)
    # absent values and values of the list go, from its middle and its ends
    has = want[(want >> np.uint64(USHIFT)) == 1]
    for cut in (has[:: max(1, has.size // k)][:k], np.concatenate([has[:2], has[-2:]]),
                _key(1, 7, np.arange(dv - 400, dv - 400 + k % 300 + 1))):
        q.stage(_batch(np.zeros(0, dtype=np.uint64), cut, dv, q.qe))
        q.transfer_update_all()
        q.transfer_update_index()
        want = np.setdiff1d(want, cut)
        assert np.array_equal(q.export(0), want)
    q.close()
    eng.close()
