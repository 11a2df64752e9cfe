"""Rows uploaded through pinned pieces by two threads: the sizes at which that
begins and ends, whole pieces and remainders.  FP32 codes that need no padding
are the rows."""

import numpy as np
import pytest

import pyglass_amd as pg

pytestmark = pytest.mark.gpu

MB_ROWS = 2048  # rows of 128 floats per MB


@pytest.mark.parametrize("n", [32 * MB_ROWS - 1, 32 * MB_ROWS, 32 * MB_ROWS + 1, 34 * MB_ROWS, 35 * MB_ROWS + 77])
def test_rows_arrive(n):
    if pg.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(n)
    rows = rng.standard_normal((n, 128)).astype(np.float32)
    # 32 ids a row: the graph is uploaded by pieces too once it is 32 MB, here it is not
    adj = np.zeros((n, 32), np.int32)
    adj[:] = np.arange(32)
    print(f"staged upload n={n}", flush=True)
    for quant, refine in (("FP32", ""), ("SQ8U", "FP32")):
        s = pg.Searcher(pg.Graph.from_arrays(adj, [0]), rows, "L2", quant, refine)
        if quant == "FP32":
            np.testing.assert_array_equal(s.codes().view(np.float32).reshape(n, 128), rows)
        else:
            assert s.calibration()[0] == rows.min()
        del s
