"""More queries than slots where the queries of some work counters take far
longer than the others': slots whose own counter is used up go on with the
queries of the rest, every query is answered once, and the counters are clear
again for the next launch.  Against the oracle."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks", [1, 3, 16, 40])
@pytest.mark.parametrize("qwaves", [1, 2])
def test_slots_take_over_from_slower_counters(blocks, qwaves):
    if pg.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(6)
    X = rng.integers(0, 256, (3000, 64)).astype(np.float32)
    adj = rng.integers(0, 3000, (3000, 24)).astype(np.int32)
    Q = rng.integers(0, 256, (600, 64)).astype(np.float32)
    s = pg.Searcher(pg.Graph.from_arrays(adj, [7]), X, "L2", "SQ8U")
    o = O.Searcher(O.Graph(adj=adj, eps=[7]), X, "L2", "SQ8U")
    want = {}
    for ef in (9, 250):
        o.set_ef(ef)
        want[ef] = o.batch_search(Q, 8)
    s.set_launch(0, 1, blocks)
    s.set_query_waves(qwaves)
    slow = {"one of sixteen": np.arange(600) % 16 == 5, "all but one": np.arange(600) % 16 != 5,
            "the first": np.arange(600) < 64, "none": np.zeros(600, bool)}
    for name, m in slow.items():
        for nq in (600, blocks + 1, 17 * blocks + 5 if blocks < 30 else 599):
            print(f"take-over blocks={blocks} qwaves={qwaves} slow={name} nq={nq}", flush=True)
            ef = np.where(m, 250, 9).astype(np.int32)[:nq]
            I, D = s.batch_search_efk(Q[:nq], ef, 8)
            Io = np.where(m[:nq, None], want[250][0][:nq], want[9][0][:nq])
            Do = np.where(m[:nq, None], want[250][1][:nq], want[9][1][:nq])
            np.testing.assert_array_equal(np.stack(I), Io)
            np.testing.assert_array_equal(np.stack(D), Do)
