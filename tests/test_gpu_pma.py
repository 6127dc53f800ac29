"""Packed-memory array deletes and list extraction at the sizes where their
kernels change: delete keys of a leaf compared one by one or by rank, more than
64 of them, whole leaves; rows that end in the 64 keys they begin in, or that
reach back over many.  Expected lists by numpy set operations."""
import numpy as np
import pytest

from cgbdsm_amd.engine import Engine
from cgbdsm_amd.host import KeyBatch, Planner

pytestmark = pytest.mark.gpu

USHIFT = 59  # ebits 5


def _key(d, u, v):
    return (np.uint64(d) << np.uint64(USHIFT)) | (np.uint64(u) << np.uint64(32)) | np.asarray(v, dtype=np.uint64)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 129, 5000])
@pytest.mark.parametrize("k", [1, 16, 17, 64, 65, 700])
def test_pma_delete_and_extract(n, k):
    print(f"case pma n={n} k={k}", flush=True)
    rng = np.random.default_rng(n * 131 + k)
    dv = 4 * n + 1000
    pl = Planner(np.array([0, 1, 2], dtype=np.int32), np.array([[0, 1], [1, 2]], dtype=np.uint32))
    eng = Engine(0)
    q = eng.query(pl.query_tables)
    q.set_layout("gpma")
    held = _key(1, 7, rng.permutation(dv)[:n].astype(np.uint64))
    short = np.concatenate([_key(d, u, rng.permutation(dv)[: rng.integers(1, 4)].astype(np.uint64))
                            for d in (0, 1, 3) for u in range(20, 60)])
    want = np.unique(np.concatenate([held, short]))
    card, avg = q.index_init(want, dv)
    q.set_plan(pl.make_plan(card, avg))
    none = np.zeros(0, dtype=np.uint64)
    assert np.array_equal(q.export(0), want)
    for cut in (want[:k], want[-k:], rng.permutation(want)[:k], _key(1, 7, np.arange(k) % dv), want):
        cut = np.unique(cut)
        q.stage(KeyBatch(0, none, cut, none, np.zeros(q.qe, dtype=np.uint8), dv, 0, {}))
        q.transfer_update_all()
        q.transfer_update_index()
        want = np.setdiff1d(want, cut)
        assert np.array_equal(q.export(0), want)
        q.stage(KeyBatch(0, held[: n // 2 + 1], none, none, np.zeros(q.qe, dtype=np.uint8), dv, 0, {}))
        q.transfer_update_all()
        q.transfer_update_index()
        want = np.union1d(want, held[: n // 2 + 1])
        assert np.array_equal(q.export(0), want)
    q.close()
    eng.close()
