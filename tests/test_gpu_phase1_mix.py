"""The database sweep of one query where a few profiles are much longer than
the rest: these go to workgroups of their own whose waves take the query's
stripes side by side.  Their maxima equal the oracle's and those of
workgroups of one wave, which have no such bands, for every number of rows per
lane, one to eleven stripes, and lengths around a refill and a hand-off ring.
With context vectors there are no bands; the same databases are checked."""
import numpy as np
import pytest
from comer2_amd._ffi import SynthDB
from comer2_amd.host import encode_key
from gpu_common import oracle, processing

pytestmark = pytest.mark.gpu

LONG = [190, 191, 192, 193, 222, 223, 224, 225, 255, 256, 257, 258, 289, 700, 1501]


def _sets(lq, nprof):
    rng = np.random.default_rng(lq)
    lens = np.concatenate([rng.integers(64, 72, nprof), np.array(LONG)])
    rng.shuffle(lens)
    q = SynthDB.from_lengths(401, [lq])
    return q, SynthDB.from_lengths(402, lens), lens


# one profile of 64-71 positions per segment; 900: 4 waves per workgroup, 2,500: 8
@pytest.mark.parametrize("nprof", [900, 2500])
@pytest.mark.parametrize("lq,rmax", [(64, 5), (65, 5), (129, 5), (223, 5), (300, 5), (321, 5), (600, 3), (700, 2),
                                     (513, 1), (700, 1), (1337, 5)])
def test_long_profiles(lq, rmax, nprof):
    q, d, lens = _sets(lq, nprof)
    print(f"long profiles: Lq={lq} rmax={rmax} nprof={nprof}", flush=True)
    cbp = processing(dict(max_map_pairs=0))
    cbp.set_tuning(4096, rmax, 8)
    cbp.TransferQueries(q)
    cbp.TransferCPMData(d)
    cbp.SetDbDetails(d.npos, d.nprof)
    keys = cbp.phase1_keys(0)
    orc = oracle()
    pick = [int(i) for i in np.flatnonzero(lens > 100)] + [int(i) for i in np.linspace(0, d.nprof - 1, 40)]
    for dp in pick:
        S, _ = orc.score_f32(q.view, 0, d.view, dp)
        m, _, _ = orc.viterbi_f32(q.view, 0, d.view, dp, S)
        assert int(keys[dp]) == encode_key(m.maxsc, m.x, m.y), (lq, rmax, dp, int(lens[dp]))
    cbp.set_tuning(4096, rmax, 1)
    assert np.array_equal(keys, cbp.phase1_keys(0))


@pytest.mark.parametrize("lq", [64, 65, 128, 129, 181, 300, 700])
def test_long_profiles_with_context_vectors(lq):
    q, d, lens = _sets(lq, 2500)
    q.add_cv(403)
    d.add_cv(404)
    opts = dict(max_map_pairs=0, cvswgt=0.15)
    keys = {}
    for rmax in (2, 1):
        print(f"long profiles, context vectors: Lq={lq} rmax={rmax}", flush=True)
        cbp = processing(opts)
        cbp.set_tuning(4096, rmax, 8)
        cbp.TransferQueries(q)
        cbp.TransferCPMData(d)
        cbp.SetDbDetails(d.npos, d.nprof)
        keys[rmax] = cbp.phase1_keys(0)
        cbp.close()
    orc = oracle(opts)
    for dp in [int(i) for i in np.flatnonzero(lens > 100)] + [int(i) for i in np.linspace(0, d.nprof - 1, 20)]:
        S, _ = orc.score_f32(q.view, 0, d.view, dp)
        m, _, _ = orc.viterbi_f32(q.view, 0, d.view, dp, S)
        assert int(keys[2][dp]) == encode_key(m.maxsc, m.x, m.y), (lq, dp, int(lens[dp]))
    assert np.array_equal(keys[2], keys[1])
