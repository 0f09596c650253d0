"""The MAP passes' rows per lane, stripes and waves for a query: the streaming
passes have one row per lane up to 1,024 rows (16 waves); the passes of a
workgroup per pair, whose bands have 8 waves, as few rows per lane as let one
band cover the query."""
import ctypes as C
import os
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("lq", [1, 64, 65, 512, 513, 640, 641, 1000, 1024, 1025, 1536, 1537, 2560, 2561, 5000])
def test_geometry(lq):
    from comer2_amd import _ffi
    _ffi.load_hip()
    T = C.CDLL(os.path.join(ROOT, "tests", "libadapter_check.so"))
    out = (C.c_int * 3)()
    for pipe in (0, 1):
        T.c2t_map_geometry(lq, pipe, out)
        rows, ns, nw = list(out)
        assert ns == -(-lq // (64 * rows))
        if pipe and lq <= 1024:
            assert rows == 1 and nw == ns <= 16
        else:
            assert rows == min(5, -(-lq // 512)) and nw == min(ns, 8)
            assert nw == ns or lq > 2560
