"""The visited set's forms against the oracle: a bitset of every row, buckets
of four 16-bit entries, buckets of two 32-bit entries, and the move to the
slot's global bitset from each, at the row counts where one form ends.
Visited sets are exact, so ids, distances and evaluation counts are equal."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")


# 256 words: a bitset up to 8,192 rows, remainders of 14 bits up to 2^21 rows,
# 32-bit entries above; 2,048 words: a bitset up to 65,536 rows
@pytest.mark.parametrize("n,words", [(1, 256), (33, 256), (8192, 256), (8193, 256), (65536, 2048), (65537, 2048),
                                     (1 << 21, 256), ((1 << 21) + 1, 256), ((1 << 21) + 1, 2048)])
def test_visited_forms_match_oracle(n, words):
    rng = np.random.default_rng(n)
    X = rng.integers(0, 256, (n, 8)).astype(np.float32)
    adj = rng.integers(0, n, (n, 16)).astype(np.int32)
    eps = [int(n // 2)]
    Q = rng.integers(0, 256, (64, 8)).astype(np.float32)
    print(f"visited n={n} words={words}", flush=True)
    s = pg.Searcher(pg.Graph.from_arrays(adj, eps), X, "L2", "SQ8U")
    o = O.Searcher(O.Graph(adj=adj, eps=eps), X, "L2", "SQ8U")
    s.set_visited_capacity(words)
    s.set_launch(0, 1, 16)  # four queries in a row on every slot
    for ef in (8, 60, 300):  # within the table, past 384 ids, past 3,072
        s.set_ef(ef)
        o.set_ef(ef)
        I, D = s.batch_search(Q, 5)
        Io, Do = o.batch_search(Q, 5)
        np.testing.assert_array_equal(I, Io)
        np.testing.assert_array_equal(D, Do)
        assert s.get_last_search_dist_cmps() == o.get_last_search_dist_cmps()
