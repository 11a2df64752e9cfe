"""k-means calls whose nearest centroids are found without the filter, on both
sides of the sizes at which the exact kernel changes its form and the filter
comes in, against the oracle.  Ids and centroids are equal."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")


@pytest.mark.parametrize("n,d,k", [(1, 1, 1), (63, 3, 2), (300, 32, 16), (1025, 4, 4), (4900, 64, 64), (5000, 64, 64),
                                   (30900, 64, 64), (31000, 64, 64), (16000, 4, 1021), (40000, 31, 66), (200, 768, 130),
                                   (1000, 200, 257), (70001, 5, 3)])
def test_small_calls_match_oracle(n, d, k):
    rng = np.random.default_rng(n + d + k)
    F = rng.standard_normal((max(n, 2 * k + 3), d)).astype(np.float32)
    print(f"k-means small n={n} d={d} k={k}", flush=True)
    c, o = pg.Clustering(k, 2), O.Clustering(k, 2, "random").fit(F)
    c.fit(F)
    np.testing.assert_array_equal(c.centroids(), o.centroids)
    X = rng.standard_normal((n, d)).astype(np.float32)
    if n > 4:
        X[1, 0], X[2, d - 1], X[3] = np.nan, -np.inf, 1e30
    np.testing.assert_array_equal(c.predict(X), o.predict(X))
