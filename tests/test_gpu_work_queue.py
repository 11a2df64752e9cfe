"""Batches of more queries than slots, handed out through 16 counters: every
query once, and the counters at zero for the next launch, whatever the
remainders of queries and slots by 16, against the oracle."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pair():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(5)
    X = rng.integers(0, 256, (3000, 64)).astype(np.float32)
    adj = rng.integers(0, 3000, (3000, 24)).astype(np.int32)
    Q = rng.integers(0, 256, (700, 64)).astype(np.float32)
    s = pg.Searcher(pg.Graph.from_arrays(adj, [7]), X, "L2", "SQ8U")
    o = O.Searcher(O.Graph(adj=adj, eps=[7]), X, "L2", "SQ8U")
    for x in (s, o):
        x.set_ef(20)
    return s, Q, o.batch_search(Q, 8)


@pytest.mark.parametrize("blocks", [1, 2, 15, 16, 17, 33, 256])
@pytest.mark.parametrize("qwaves", [1, 4])  # a wave per query, four on each
def test_every_query_once(pair, blocks, qwaves):
    s, Q, (Io, Do) = pair
    s.set_query_waves(qwaves)
    s.set_launch(0, 1, blocks)
    for nq in (blocks, blocks + 1, 2 * blocks + 15, 31 * (blocks < 17) + blocks, 700):
        print(f"queue blocks={blocks} qwaves={qwaves} nq={nq}", flush=True)
        I, D = s.batch_search(Q[:nq], 8)
        np.testing.assert_array_equal(I, Io[:nq])
        np.testing.assert_array_equal(D, Do[:nq])
