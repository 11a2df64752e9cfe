"""k-means kernels at the edges of their tiles, against the oracle: rows not a
multiple of 64, centroids around multiples of 256 and split over workgroups,
dimensions around multiples of 16 and 256, and rows that the matrix-core
filter cannot decide (ties, tiny and huge values, infinities, NaN), which the
exact kernel answers.  Ids and centroids are equal."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")


def both(X, k, epochs):
    c = pg.Clustering(k, epochs)
    c.fit(X)
    o = O.Clustering(k, epochs, "random").fit(X)
    np.testing.assert_array_equal(c.centroids(), o.centroids)
    return c, o


@pytest.mark.parametrize("n,d,k", [(3, 1, 1), (65, 3, 63), (700, 15, 255), (700, 16, 256), (700, 17, 257), (3000, 33, 513),
                                   (1500, 255, 40), (1500, 257, 40), (600, 530, 7), (5000, 8, 1100)])
def test_fit_and_predict_match_oracle(n, d, k):
    rng = np.random.default_rng(n + d + k)
    X = rng.standard_normal((n, d)).astype(np.float32)
    print(f"k-means n={n} d={d} k={k}", flush=True)
    c, o = both(X, k, 3)
    np.testing.assert_array_equal(c.predict(X), o.predict(X))
    np.testing.assert_array_equal(c.predict(X[:1]), o.predict(X[:1]))


def test_random_seeding_needs_more_sampled_rows_than_clusters():
    # drawing k of k sampled rows divides by zero in the reference
    with pytest.raises(pg.GlassError):
        pg.Clustering(1, 3).fit(np.zeros((2, 1), np.float32))


def test_undecided_rows_match_oracle():
    rng = np.random.default_rng(5)
    base = rng.integers(-2, 3, (40, 24)).astype(np.float32)
    X = base[rng.integers(0, 40, 4000)]  # few distinct rows: equal centroids and equal distances
    print("k-means undecided rows", flush=True)
    c, o = both(X, 300, 2)
    P = np.concatenate([X[:200], X[:50] * np.float32(1e-20), X[:50] * np.float32(1e18), X[:50] * np.float32(1e30),
                        X[:10]]).astype(np.float32)
    P[-10:-5, 3] = np.nan
    P[-5:, 7] = np.inf
    np.testing.assert_array_equal(c.predict(P), o.predict(P))
    tiny = (X * np.float32(1e-25)).astype(np.float32)  # every squared norm underflows
    c, o = both(tiny, 20, 2)
    np.testing.assert_array_equal(c.predict(tiny), o.predict(tiny))


def test_skewed_clusters_and_pieces_match_oracle():
    """One cluster of most rows (its list is emptied many times), and a
    predict whose rows go to the device in several pieces."""
    rng = np.random.default_rng(9)
    X = rng.standard_normal((30000, 300)).astype(np.float32) * np.float32(0.01)
    X[:40] += 100
    print("k-means skewed", flush=True)
    c, o = both(X, 3, 2)
    np.testing.assert_array_equal(c.predict(X), o.predict(X))
