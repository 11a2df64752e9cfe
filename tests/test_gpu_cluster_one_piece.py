"""predict() around the sizes at which its rows begin to go to the device in
pieces (24 MB) and in more of them, against the oracle.  Ids are equal."""

import numpy as np
import pytest

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [32768, 32769, 49151, 49152, 49153, 65536, 65537])
def test_rows_around_a_piece(n):
    if pg.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 128)).astype(np.float32)
    print(f"predict pieces n={n}", flush=True)
    c, o = pg.Clustering(20, 2), O.Clustering(20, 2, "random").fit(X[:500])
    c.fit(X[:500])
    np.testing.assert_array_equal(c.predict(X), o.predict(X))
