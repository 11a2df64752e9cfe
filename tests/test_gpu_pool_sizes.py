"""Pools around the sizes where the merge changes (one chunk of 64 entries, two,
four, and LDS) against the oracle, with many equal distances: ids, distances
and their order are those of inserting one neighbour at a time."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")


@pytest.mark.parametrize("quant", ["SQ8U", "SQ4U", "FP32"])
@pytest.mark.parametrize("qwaves", [1, 2])
def test_pools_match_oracle(quant, qwaves):
    rng = np.random.default_rng(11)
    X = rng.integers(0, 4, (2500, 24)).astype(np.float32)  # few distinct distances
    adj = rng.integers(0, 2500, (2500, 32)).astype(np.int32)
    adj[rng.random((2500,)) < 0.3, 20:] = -1
    Q = rng.integers(0, 4, (40, 24)).astype(np.float32)
    s = pg.Searcher(pg.Graph.from_arrays(adj, [3]), X, "L2", quant)
    o = O.Searcher(O.Graph(adj=adj, eps=[3]), X, "L2", quant)
    s.set_query_waves(qwaves)
    for ef, k in ((1, 1), (15, 16), (48, 10), (63, 63), (64, 1), (10, 64), (65, 10), (80, 81), (128, 10), (129, 129),
                  (256, 20), (257, 5)):
        print(f"pool {quant} qwaves={qwaves} ef={ef} k={k}", flush=True)
        s.set_ef(ef)
        o.set_ef(ef)
        I, D = s.batch_search(Q, k)
        Io, Do = o.batch_search(Q, k)
        np.testing.assert_array_equal(I, Io)
        np.testing.assert_array_equal(D, Do)
