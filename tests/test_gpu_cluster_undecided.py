"""Many rows that the nearest-centroid filter cannot decide: few centroids are
distinct, so the rows near the equal ones go to the exact kernel, which takes
them one to a workgroup or 64 to a workgroup by their number.  Ids equal the
oracle's."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")


# dimensions with every tail (8 + 4 + 1, 8 + 3, none), centroids of every
# remainder by four; the forms change at about 11,570, 11,270 and 13,900 rows
@pytest.mark.parametrize("d,k,counts", [(133, 513, (0, 1, 63, 64, 65, 1025, 11500, 11640, 20000)),
                                        (75, 1030, (11200, 11350, 20000)), (768, 19, (13850, 13950, 20000))])
def test_undecided_rows_match_oracle(d, k, counts):
    rng = np.random.default_rng(d)
    points = (100 * rng.standard_normal((max(2, k // 2), d))).astype(np.float32)
    X = points[rng.integers(0, len(points), 8 * k)]
    c, o = pg.Clustering(k, 1), O.Clustering(k, 1, "random").fit(X)  # empty clusters: zero centroids
    c.fit(X)
    np.testing.assert_array_equal(c.centroids(), o.centroids)
    P = (points[rng.integers(0, len(points), 20000)] + rng.standard_normal((20000, d))).astype(np.float32)
    P[-1, 0], P[-2, 1] = np.nan, np.inf
    at = rng.permutation(19990)
    near = (0.01 * rng.standard_normal((20000, d))).astype(np.float32)
    clear, tied = o.predict(P), o.predict(near)
    for n in counts:
        print(f"undecided d={d} k={k} rows={n}", flush=True)
        T, want = P.copy(), clear.copy()
        T[at[:n]], want[at[:n]] = near[at[:n]], tied[at[:n]]
        np.testing.assert_array_equal(c.predict(T), want)
