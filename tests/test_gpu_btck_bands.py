"""The backtrack pass of queries of several stripes: a candidate's stripes run
side by side in a band of up to four waves, in rounds, and give the records
and alignments of one wave taking the stripes in turn (the host-decided
lists), bit for bit; profile lengths around a refill, the waves' distance and
a hand-off ring, 2 to 5 stripes and more, 1 to 4 rows per lane (a query of
several stripes has no more), and more candidates than workgroups."""
import numpy as np
import pytest
from comer2_amd._ffi import SynthDB
from gpu_common import processing

pytestmark = pytest.mark.gpu

EDGES = [3, 4, 31, 32, 33, 34, 62, 63, 64, 65, 66, 94, 95, 96, 97, 98, 127, 128, 129, 200, 391]


# (query length, most rows per lane, copies of the list): 2, 3, 4, 5, 6, 9 and
# 13 stripes
@pytest.mark.parametrize("lq,rmax,copies", [(65, 1, 1), (192, 1, 2), (250, 1, 1), (258, 1, 1), (577, 1, 1),
                                            (300, 2, 1), (780, 2, 1), (600, 3, 1), (321, 5, 60), (1337, 5, 20),
                                            (700, 5, 1), (3000, 5, 1)])
def test_bands_equal_one_wave(lq, rmax, copies):
    q = SynthDB.from_lengths(301, [lq])
    d = SynthDB.from_lengths(302, EDGES * copies + [900, 1500])
    d.plant(q, 303, 8, 3.0, 60.0)
    cbp = processing(dict(mapaln=0, max_map_pairs=0))
    cbp.set_tuning(4096, rmax, 8)
    cbp.TransferQueries(q)
    cbp.TransferCPMData(d)
    cbp.SetDbDetails(d.npos, d.nprof)
    out = {}
    for dev in (False, True):
        cbp.set_device_lists(dev)
        print(f"backtrack bands: Lq={lq} rmax={rmax} copies={copies} device={dev}", flush=True)
        out[dev] = cbp.ProcessScoreMatrix(0, scorethld=-1.0, logevthld=50.0)
    assert cbp.last_fallbacks() == 0
    a, b = out[False], out[True]
    assert a["npassed"] == b["npassed"] >= len(EDGES) * copies // 2 and a["nmap"] == b["nmap"] > 0
    for k in ("alndata", "order", "aln_raw"):
        assert np.ascontiguousarray(a[k]).tobytes() == np.ascontiguousarray(b[k]).tobytes(), k
