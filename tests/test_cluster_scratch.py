"""Device scratch of the nearest-centroid sweep: predict() reserves it once for
its longest piece of rows and lays it out for every piece, so the layout for
fewer rows must stay within what was reserved for more, though fewer rows are
split over more workgroups.  Address arithmetic of the built library, on the
CPU."""

import ctypes

import pytest

import pyglass_amd._lib as _lib

ROUND = 64  # rows per workgroup


class Scratch(ctypes.Structure):
    # AssignScratch: x2 and list of n words, c2 of k, m1, m2 and i1 of splits * n, two single words
    _fields_ = [(f, ctypes.c_void_p) for f in ("x2", "c2", "m1", "m2", "i1", "list", "count", "c2max")]


def end_of(lib, n, k):
    """Bytes from the scratch's start to the end of its last array, for n rows."""
    base = 1 << 20
    s = Scratch()
    place = lib._ZN9glass_hip13AssignScratch5placeEPvii
    place.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int32, ctypes.c_int32]
    place.restype = None
    place(ctypes.byref(s), base, n, k)
    assert s.x2 == base and s.c2 - s.x2 == 4 * n and s.m1 - s.c2 == 4 * k
    part = s.m2 - s.m1
    assert part % (4 * n) == 0 and part >= 4 * n and s.i1 - s.m2 == part and s.list - s.i1 == part
    assert s.count - s.list == 4 * n and s.c2max - s.count == 4
    return s.c2max + 4 - base


@pytest.mark.parametrize("d,k", [(16, 1000), (64, 512), (64, 513), (96, 1000), (128, 600), (128, 1024), (200, 5000),
                                 (300, 3), (960, 4100), (4096, 70000), (100000, 20000)])
def test_scratch_for_more_rows_holds_every_piece(d, k):
    lib = _lib.load()
    size = lib._ZN9glass_hip13AssignScratch5bytesEii
    size.argtypes = [ctypes.c_int32, ctypes.c_int32]
    size.restype = ctypes.c_size_t
    piece = max(ROUND, (4 << 20) // d // ROUND * ROUND)  # rows of predict's full piece
    for n in (piece, piece - 1, piece // 2 + 1, 4096, 65, 1):
        have = size(n, k)
        rows = set(range(1, min(n, 300) + 1)) | set(range(max(1, n - 300), n + 1)) | set(range(1, n + 1, 61))
        rows |= set(range(ROUND, n + 1, ROUND)) | {r - 1 for r in range(ROUND, n + 1, ROUND)}
        over = [(c, end_of(lib, c, k) - have) for c in sorted(rows) if end_of(lib, c, k) > have]
        assert not over, f"{n} rows reserved, k {k}: {len(over)} shorter pieces run over, first {over[0]}, last {over[-1]}"
