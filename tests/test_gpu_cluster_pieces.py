"""predict() over several pieces of rows whose last piece is shorter than the
others and split over more workgroups than they are, against the oracle.  Ids
are equal."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")


@pytest.mark.parametrize("n,d,k", [(131008, 64, 520), (65472, 128, 600), (32768 + 4033, 128, 1030)])
def test_short_last_piece_matches_oracle(n, d, k):
    rng = np.random.default_rng(n + k)
    X = rng.standard_normal((n, d)).astype(np.float32)
    print(f"k-means pieces n={n} d={d} k={k}", flush=True)
    c, o = pg.Clustering(k, 1), O.Clustering(k, 1, "random").fit(X[:5000])
    c.fit(X[:5000])
    np.testing.assert_array_equal(c.centroids(), o.centroids)
    np.testing.assert_array_equal(c.predict(X), o.predict(X))
