"""Visited sets of large id ranges: 16- and 32-bit table entries, ids of up to
24 bits and more (each has its own multiplication), the largest remainders
(fewest displacements), and queries that stay in the table, leave it and fill
it at once.  A small graph's nodes are spread over the rows of a large one, so
the oracle searches the small one: neighbours, distances and evaluation counts
are the same."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NODES, K = 4000, 24


@pytest.fixture(scope="module")
def small():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(12)
    X = rng.standard_normal((NODES, 4)).astype(np.float32)
    adj = rng.integers(0, NODES, (NODES, K)).astype(np.int32)
    adj[::7, K - 5:] = -1
    Q = rng.standard_normal((90, 4)).astype(np.float32)
    o = O.Searcher(O.Graph(adj=adj, eps=[5]), X, "L2", "FP32")
    want = {}
    for ef in (10, 40, 150):
        o.set_ef(ef)
        want[ef] = o.batch_search(Q, 10)
    return X, adj, Q, want


# rows, words: (bits of an id, of a remainder, of an entry)
@pytest.mark.parametrize("n,words", [((1 << 21), 256),        # 21, 14, 16
                                     ((1 << 21) + 1, 256),    # 22, 15, 32
                                     ((1 << 24), 2048),       # 24, 14, 16
                                     ((1 << 24) + 1, 2048),   # 25, 15, 32
                                     ((1 << 24) + 1, 4096),   # 25, 14, 16
                                     (1 << 18, 1024),         # 18, 9, 16
                                     (70001, 256),            # 17, 10, 16
                                     (8192, 256)])            # a bitset of every row
def test_large_ids_match_the_small_graph(small, n, words):
    X, adj, Q, want = small
    rng = np.random.default_rng(n % 1009 + words)
    at = rng.permutation(min(n, 1 << 20))[:NODES].astype(np.int64) * (n // min(n, 1 << 20))
    at[0], at[1] = n - 1, n - 2  # the last rows
    at = np.unique(at)
    at = rng.permutation(np.concatenate([at, np.setdiff1d(np.arange(NODES), at)[:NODES - at.size]]))
    assert np.unique(at).size == NODES
    big = np.zeros((n, 4), np.float32)
    big[at] = X
    rows = np.full((n, K), -1, np.int32)
    rows[at] = np.where(adj < 0, -1, at[adj])
    s = pg.Searcher(pg.Graph.from_arrays(rows, [int(at[5])]), big, "L2", "FP32")
    s.set_visited_capacity(words)
    for qwaves in (1, 2):
        s.set_query_waves(qwaves)
        for ef in (10, 40, 150):
            print(f"visited forms n={n} words={words} qwaves={qwaves} ef={ef}", flush=True)
            s.set_ef(ef)
            Io, Do = want[ef]
            for _ in range(2):  # the slots' bitsets are clear again
                I, D = s.batch_search(Q, 10)
                np.testing.assert_array_equal(I, at[Io])
                np.testing.assert_array_equal(D, Do)
