"""The streaming MAP passes at the edges of their schedule.

They work in groups of four steps, move a profile's transitions in blocks of
64 columns and take queries of up to 1,024 rows as one band of up to 16
waves: profile lengths around a group and a block, and query lengths around
a wave, the two old and new band limits, give the oracle's alignments and
what the per-pair kernels give, bit for bit.
"""
import numpy as np
import pytest
from comer2_amd._ffi import SynthDB
from gpu_common import oracle, processing

pytestmark = pytest.mark.gpu

ED = [5, 6, 7, 8, 9, 62, 63, 64, 65, 66, 126, 127, 128, 129, 130, 257]


def _run(q, d, pipe):
    cbp = processing(dict(max_map_pairs=0))
    cbp.set_map_pipe(pipe)
    cbp.TransferQueries(q)
    cbp.TransferCPMData(d)
    cbp.SetDbDetails(d.npos, d.nprof)
    res = cbp.ProcessScoreMatrix(0, scorethld=-1.0, logevthld=50.0)
    cbp.close()
    return res


@pytest.mark.parametrize("lq", [5, 63, 64, 65, 511, 512, 513, 960, 961, 1023, 1024, 1025])
def test_map_band_edges(lq):
    q = SynthDB.from_lengths(141, [lq])
    d = SynthDB.from_lengths(142, ED)
    print(f"map band edges: Lq={lq}", flush=True)
    res = _run(q, d, True)
    per = _run(q, d, False)
    for k in ("alndata", "order", "aln_raw"):
        a, b = np.ascontiguousarray(res[k]), np.ascontiguousarray(per[k])
        assert a.tobytes() == b.tobytes(), (lq, k)
    orc = oracle()
    sel = [int(i) for i in res["order"] if res["logE"][i] <= 50.0]
    assert list(res["map_rows"]) == sel and sel
    for k, row in enumerate(sel):
        dp = int(res["pronr"][row])
        S, M = orc.score_f32(q.view, 0, d.view, dp)
        r, _, _, _, aln = orc.map(q.view, 0, d.view, dp, S, M, np.float32(res["epa"][row]))
        ctx = (lq, ED[dp])
        assert res["alnlen"][row] == r.alnlen, ctx
        assert res["beg"][row] == ((r.begx << 16) | r.begy), ctx
        assert res["end"][row] == ((r.x << 16) | r.y), ctx
        got = tuple(res["alns"][k])
        assert got == tuple(bytes(aln[j]).split(b"\0")[0].decode() for j in range(3)), ctx
