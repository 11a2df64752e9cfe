"""Host calls against the oracle over the sizes of their buffers: those the
kernel reads and writes in pinned host memory (to 2 MiB of queries, results and
counters), and those copied, with arrays that do not end on 16 bytes."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def searchers():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(3)
    X = rng.integers(0, 256, (2000, 37)).astype(np.float32)
    adj = rng.integers(0, 2000, (2000, 16)).astype(np.int32)
    s = pg.Searcher(pg.Graph.from_arrays(adj, [5]), X, "L2", "SQ8U", "FP32")
    o = O.Searcher(O.Graph(adj=adj, eps=[5]), X, "L2", "SQ8U", "FP32")
    for x in (s, o):
        x.set_ef(12)
    return s, o


# 240 bytes a query: 8,738 queries are the last that fit 2 MiB.  In turn, so
# that the buffers shrink, grow and change kind from one call to the next.
@pytest.mark.parametrize("nq", [1, 3, 8738, 8739, 2, 8737])
def test_host_batches_match_oracle(searchers, nq):
    s, o = searchers
    Q = np.random.default_rng(nq).integers(0, 256, (nq, 37)).astype(np.float32)
    print(f"host call nq={nq}", flush=True)
    I, D = s.batch_search(Q, 10)
    Io, Do = o.batch_search(Q, 10)
    np.testing.assert_array_equal(I, Io)
    np.testing.assert_array_equal(D, Do)
    assert s.get_last_search_dist_cmps() == o.get_last_search_dist_cmps()
    # per-query ef and k: each query's answer is that of a call of its own
    m = min(nq, 60)
    ef, k = np.arange(m) % 13 + 4, np.arange(m) % 9 + 1
    I, D, cnt = s.batch_search_efk(Q[:m], ef, k, with_counters=True)
    for i in range(m):
        Ii, Di = o.batch_search(Q[i:i + 1], int(k[i]), ef=int(ef[i]))
        np.testing.assert_array_equal(I[i], Ii[0])
        np.testing.assert_array_equal(D[i], Di[0])
        assert cnt[i, 0] == o.last_counts[0][0]
