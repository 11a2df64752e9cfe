"""Row distances at the edges of their batches, against the oracle: dimensions
whose steps of 16 fill a batch, pass it by one or leave a remainder, and graph
degrees that give an expansion 1 to 64 new neighbours, so that rows are shared
by 4, 8 and 16 lanes and by two rows per lane group, and integer rows take one
and several passes.  One wave per query and four; ids, distances and
evaluation counts are equal."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")


def graph(n, degree, rng):
    adj = rng.integers(0, n, (n, degree)).astype(np.int32)
    for i in range(n):  # rows of every length, and a way round
        adj[i, 0] = (i + 1) % n
        adj[i, 1 + i % degree:] = -1
    return adj


@pytest.mark.parametrize("dim", [16, 31, 100, 128, 255, 260, 272, 528, 1040])
@pytest.mark.parametrize("quant,metric", [("FP32", "L2"), ("FP16", "IP"), ("BF16", "L2"), ("E5M2", "IP"), ("E5M2", "L2"),
                                          ("SQ8", "L2"), ("SQ8", "IP"), ("SQ8U", "L2"), ("SQ4U", "L2"), ("SQ2U", "L2")])
def test_row_shapes_match_oracle(dim, quant, metric):
    rng = np.random.default_rng(dim)
    n = 700
    X = rng.standard_normal((n, dim)).astype(np.float32)
    Q = rng.standard_normal((24, dim)).astype(np.float32)
    adj = graph(n, 64, rng)
    refine = "FP32" if quant in ("SQ4U", "SQ8") else ""
    print(f"rows dim={dim} {quant} {metric}", flush=True)
    s = pg.Searcher(pg.Graph.from_arrays(adj, [5]), X, metric, quant, refine)
    o = O.Searcher(O.Graph(adj=adj, eps=[5]), X, metric, quant, refine)
    for waves in (1, 4):
        s.set_query_waves(waves)
        for ef in (20, 140):  # the common and the general path
            s.set_ef(ef)
            o.set_ef(ef)
            I, D = s.batch_search(Q, 10)
            Io, Do = o.batch_search(Q, 10)
            np.testing.assert_array_equal(I, Io)
            np.testing.assert_array_equal(D, Do)
            assert s.get_last_search_dist_cmps() == o.get_last_search_dist_cmps()
            a, b = s.search(Q[0], 10)
            c, d = o.search(Q[0], 10)
            np.testing.assert_array_equal(a, c)
            np.testing.assert_array_equal(b, d)
