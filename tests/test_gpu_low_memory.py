"""A batch for whose slot areas device memory does not suffice runs on as many
slots as there is room for, with the results of the full launch."""

import numpy as np
import pytest
import torch

import pyglass_amd as pg

pytestmark = pytest.mark.gpu

N = 8_000_000  # a slot is 1 MB and its dirty list
LINKED = 200_000


def test_fewer_slots_where_memory_is_short():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(4)
    adj = np.full((N, 8), -1, np.int32)
    at = np.arange(LINKED) * (N // LINKED)
    adj[at] = at[rng.integers(0, LINKED, (LINKED, 8))]
    X = np.zeros((N, 4), np.float32)
    X[at] = rng.integers(0, 256, (LINKED, 4))
    q = torch.from_numpy(rng.integers(0, 256, (6000, 4)).astype(np.float32)).cuda()
    ids = torch.empty((6000, 10), dtype=torch.int32, device="cuda")
    cnt = torch.empty((6000, 3), dtype=torch.int32, device="cuda")
    s = pg.Searcher(pg.Graph.from_arrays(adj, [0]), X, "L2", "SQ8U")
    s.set_ef(64)
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    held = torch.empty(free - (3 << 30), dtype=torch.uint8, device="cuda")
    out = []
    try:
        for nq in (6000, 100, 6000):
            print(f"low memory nq={nq}", flush=True)
            s.search_batch_dev(q.data_ptr(), nq, 10, ids.data_ptr(), 0, cnt.data_ptr())
            s.sync()
            shape = s.get_launch()
            out.append((nq, shape["blocks"] * shape["waves_per_block"], ids[:nq].cpu().numpy(), cnt[:nq].cpu().numpy()))
    finally:
        del held
        torch.cuda.empty_cache()
    full = pg.Searcher(pg.Graph.from_arrays(adj, [0]), X, "L2", "SQ8U")
    full.set_ef(64)
    full.search_batch_dev(q.data_ptr(), 6000, 10, ids.data_ptr(), 0, cnt.data_ptr())
    full.sync()
    shape = full.get_launch()
    assert out[0][1] < shape["blocks"] * shape["waves_per_block"]  # the room was short
    for nq, waves, i, c in out:
        assert waves >= min(nq, 1000)
        np.testing.assert_array_equal(i, ids[:nq].cpu().numpy())
        np.testing.assert_array_equal(c, cnt[:nq].cpu().numpy())
