"""A server made while the searcher's own stream has work queued: its first
batches hand out every query once (their work counters are clear before they
start), and so do the ones after them."""

import threading

import numpy as np
import pytest
import torch

import pyglass_amd as pg
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def test_first_batches_of_a_server_beside_a_busy_searcher():
    if pg.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(8)
    X = rng.integers(0, 256, (3000, 64)).astype(np.float32)
    adj = rng.integers(0, 3000, (3000, 24)).astype(np.int32)
    Q = rng.integers(0, 256, (700, 64)).astype(np.float32)
    s = pg.Searcher(pg.Graph.from_arrays(adj, [7]), X, "L2", "SQ8U")
    o = O.Searcher(O.Graph(adj=adj, eps=[7]), X, "L2", "SQ8U")
    for x in (s, o):
        x.set_ef(40)
    Io, Do = o.batch_search(Q, 8)
    s.set_launch(0, 1, 16)  # 16 queries at a time: the others are handed out
    q = torch.from_numpy(Q).cuda()
    ids = torch.empty((700, 8), dtype=torch.int32, device="cuda")
    started, made = threading.Event(), threading.Event()

    def keep_busy():
        for _ in range(300):
            s.search_batch_dev(q.data_ptr(), 700, 8, ids.data_ptr())
            started.set()
            if made.is_set():
                break

    t = threading.Thread(target=keep_busy)
    t.start()
    started.wait()
    print("server beside a busy searcher", flush=True)
    srv = pg.Server(s, max_batch=700, max_k=8, max_inflight=3)
    try:
        for _ in range(3):
            tickets = [srv.submit(Q, k=8, ef=40) for _ in range(4)]
            for ticket in tickets:
                I, D = srv.wait(ticket)
                np.testing.assert_array_equal(I, Io)
                np.testing.assert_array_equal(D, Do)
    finally:
        made.set()
        t.join()
        s.sync()
        srv.close()
    np.testing.assert_array_equal(ids.cpu().numpy(), Io)
