"""Waves per query of a small batch that nothing has tuned: SQ6 and PQ8 share a
query among waves only where a node has more neighbours than one wave's 16 per
pass.  Results are the oracle's either way."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quant,dim,degree,waves", [("SQ6", 40, 16, 1), ("SQ6", 40, 32, 1), ("SQ6", 200, 32, 2),
                                                    ("SQ6", 40, 40, 2), ("PQ8", 32, 16, 1), ("PQ8", 32, 20, 2)])
def test_untuned_waves_per_query(quant, dim, degree, waves):
    if pg.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(dim + degree)
    X = rng.integers(0, 256, (2000, dim)).astype(np.float32)
    adj = rng.integers(0, 2000, (2000, degree)).astype(np.int32)
    Q = rng.integers(0, 256, (20, dim)).astype(np.float32)
    s = pg.Searcher(pg.Graph.from_arrays(adj, [3]), X, "L2", quant)
    o = O.Searcher(O.Graph(adj=adj, eps=[3]), X, "L2", quant)
    s.set_ef(50)
    o.set_ef(50)
    print(f"untuned waves {quant} dim={dim} degree={degree}", flush=True)
    I, D = s.batch_search(Q, 10)
    assert s.get_query_waves()[0] == waves
    Io, Do = o.batch_search(Q, 10)
    np.testing.assert_array_equal(I, Io)
    np.testing.assert_array_equal(D, Do)


def test_tuning_keeps_eight_waves_of_wide_rows():
    """optimize() tries at most 4 waves per query; where it takes 4, wide rows
    still get 8 in batches that leave room for them."""
    if pg.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(8)
    X = rng.standard_normal((3000, 832)).astype(np.float32)
    adj = rng.integers(0, 3000, (3000, 32)).astype(np.int32)
    Q = rng.standard_normal((4, 832)).astype(np.float32)
    s = pg.Searcher(pg.Graph.from_arrays(adj, [3]), X, "L2", "SQ8")
    o = O.Searcher(O.Graph(adj=adj, eps=[3]), X, "L2", "SQ8")
    s.set_ef(30)
    o.set_ef(30)
    print("waves per query: untuned, tuned", flush=True)
    s.batch_search(Q, 10)
    assert s.get_query_waves()[0] == 8
    s.optimize()
    I, D = s.batch_search(Q, 10)
    last, tuned = s.get_query_waves()
    assert last == (8 if tuned == 4 else tuned)
    Io, Do = o.batch_search(Q, 10)
    np.testing.assert_array_equal(I, Io)
    np.testing.assert_array_equal(D, Do)
