"""Batched product-suffix steps over long lists: a step that reaches its entry
budget ends early and goes on at the next sibling, whose candidate range other
wavefronts may take over at any candidate.  Counts against the oracle, from
the depth-2 seeds and from the rows of the BFS levels."""
import pytest

from cgbdsm_amd.engine import Engine
from cgbdsm_amd.host import HostSession, synth_spec
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
