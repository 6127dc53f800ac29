"""Key sets of a batch at the sizes where their kernels change: up to 64 keys
(one wavefront), up to 4096 (one block), more (tiles).  M, U and M after the
commit against the oracle's index, with repeated keys in every set."""
import numpy as np
import pytest

from cgbdsm_amd.engine import Engine
from cgbdsm_amd.host import KeyBatch, Planner
from tests import oracle_lib as O

pytestmark = pytest.mark.gpu

USHIFT = np.uint64(59)  # ebits 5


def _keys(rng, n, ndir, dv):
    """n keys, a third of them on two hub rows, some of them twice."""
    d = rng.integers(0, ndir, n).astype(np.uint64)
    u = np.where(rng.random(n) < 0.3, 3, rng.integers(0, dv, n)).astype(np.uint64)
    v = rng.integers(0, dv, n).astype(np.uint64)
    k = (d << USHIFT) | (u << np.uint64(32)) | v
    k[n // 2: n // 2 + n // 8] = k[: n // 8]
    return k


@pytest.mark.parametrize("layout", ["gamma", "gpma"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1025, 4095, 4096, 4097, 9000])
def test_key_sets(n, layout):
    print(f"case key sets n={n} {layout}", flush=True)
    rng = np.random.default_rng(n)
    dv = 3000
    pl = Planner(np.array([0, 1, 2, 0], dtype=np.int32), np.array([[0, 1], [1, 2], [2, 3]], dtype=np.uint32))
    eng = Engine(0)
    q = eng.query(pl.query_tables)
    q.set_layout(layout)
    first = _keys(rng, 5000, q.ndir, dv)
    card, avg = q.index_init(first, dv)
    q.set_plan(pl.make_plan(card, avg))
    idx = O.Index(q.ndir, 5)
    idx.set_dv(dv)
    idx.init(first)
    ok = np.ones(q.qe, dtype=np.uint8)
    for _ in range(3):
        ins, upd = _keys(rng, n, q.ndir, dv), _keys(rng, n, q.ndir, dv)
        dele = np.concatenate([upd[: n // 2 + 1], rng.choice(first, n // 2)])
        q.stage(KeyBatch(0, ins, dele, upd, ok, dv, 0, {}))
        q.transfer_update_all()
        idx.insert(ins)
        idx.remove(dele)
        assert np.array_equal(q.export(0), idx.export(0))
        assert q.transfer_update_index()
        idx.rebuild_update(upd)
        assert np.array_equal(q.export(1), idx.export(1))
        q.batch_update_global_index()
        idx.insert(upd)
        assert np.array_equal(q.export(0), idx.export(0))
    q.close()
    eng.close()
