"""The no-alloc entry point's scratch array, used by one searcher after
another: slots of equal size whose dirty lists differ in length (the list is
shorter above 64M rows) must not be read with the other's layout.  Results
equal the same searcher's with scratch of its own."""

import numpy as np
import pytest
import torch

import pyglass_amd as pg

pytestmark = pytest.mark.gpu

# 16,384 + 2,087,992 words and 4,096 + 2,100,280
N1, N2 = 66_815_648, 67_208_864
LINKED = 300_000  # rows with neighbours; the others are only counted


def test_searchers_of_one_stride_and_two_layouts():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(3)
    adj = np.full((N2, 4), -1, np.int32)
    adj[:LINKED] = rng.integers(0, LINKED, (LINKED, 4))
    X = np.zeros((N2, 4), np.float32)
    X[:LINKED] = rng.integers(0, 256, (LINKED, 4))
    Q = rng.integers(0, 256, (64, 4)).astype(np.float32)
    q = torch.from_numpy(Q).cuda()
    for n in (N1, N2):
        print(f"no-alloc layout n={n}", flush=True)
        s = pg.Searcher(pg.Graph.from_arrays(adj[:n], [7]), X[:n], "L2", "SQ8U")
        s.set_ef(4096)
        s.set_visited_capacity(256)  # the queries go on in their slots' bitsets
        ids = torch.empty((64, 10), dtype=torch.int32, device="cuda")
        cnt = torch.empty((64, 3), dtype=torch.int32, device="cuda")
        s.search_batch_dev_noalloc(q.data_ptr(), 64, 10, ids.data_ptr(), 0, cnt.data_ptr())
        s.sync()
        I, D, C = s.batch_search_efk(Q, 4096, 10, with_counters=True)
        assert C[:, 0].min() > 8000  # more words set than the shorter list holds
        np.testing.assert_array_equal(cnt.cpu().numpy(), C)
        np.testing.assert_array_equal(ids.cpu().numpy(), np.stack(I))
        del s
