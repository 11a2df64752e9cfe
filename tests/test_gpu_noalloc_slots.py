"""The no-alloc entry point's scratch array is of a fixed size, so what a slot
holds beside its bitset decides how many waves search: as many slots as with
dirty lists of 4,096 words, and the results of the allocating entry point."""

import numpy as np
import pytest
import torch

import pyglass_amd as pg

pytestmark = pytest.mark.gpu

ARRAY = (128 << 20) - 256  # bytes of slot areas


@pytest.mark.parametrize("n", [100_000, 1 << 21, (1 << 21) + 1, 2_300_000])
def test_slots_of_the_array(n):
    if pg.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(n)
    adj = np.full((n, 8), -1, np.int32)
    adj[:50000] = rng.integers(0, 50000, (50000, 8)) * (n // 50000)
    adj[np.arange(50000) * (n // 50000)] = adj[:50000].copy()
    X = rng.integers(0, 256, (n, 4)).astype(np.float32)
    s = pg.Searcher(pg.Graph.from_arrays(adj, [0]), X, "L2", "SQ8U")
    s.set_ef(300)
    s.set_visited_capacity(256)  # the queries go on in their slots' bitsets
    q = torch.from_numpy(rng.integers(0, 256, (3000, 4)).astype(np.float32)).cuda()
    out = []
    for call in (s.search_batch_dev, s.search_batch_dev_noalloc, s.search_batch_dev_noalloc):
        print(f"no-alloc slots n={n}", flush=True)
        ids = torch.empty((3000, 10), dtype=torch.int32, device="cuda")
        cnt = torch.empty((3000, 3), dtype=torch.int32, device="cuda")
        call(q.data_ptr(), 3000, 10, ids.data_ptr(), 0, cnt.data_ptr())
        s.sync()
        out.append((ids.cpu().numpy(), cnt.cpu().numpy()))
        shape = s.get_launch()
    for ids, cnt in out[1:]:
        np.testing.assert_array_equal(ids, out[0][0])
        np.testing.assert_array_equal(cnt, out[0][1])
    fit = ARRAY // (4 * (4096 + (-(-n // 32) + 3) // 4 * 4))
    assert shape["blocks"] * shape["waves_per_block"] >= min(3000, fit) // shape["waves_per_block"] * shape["waves_per_block"]
