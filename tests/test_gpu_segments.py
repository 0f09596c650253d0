"""Phase-1 segments and waves per workgroup chosen from the chunk's size: the
maxima equal the oracle's at the counts where the launch shape changes, for
databases in any order, and a batch's queue equals the one-query launches."""
import numpy as np
import pytest
from comer2_amd._ffi import SynthDB
from gpu_common import expected_keys, oracle, processing

pytestmark = pytest.mark.gpu


# 1, 2, 4 and 8 waves per workgroup start at 1, 257, 513 and 1,025 segments
# (one profile each here), on both sides of each line; one and two stripes
@pytest.mark.parametrize("nprof,qlen", [(n, 37) for n in (1, 3, 256, 257, 512, 513, 1024, 1025)] +
                         [(n, 333) for n in (1, 3, 257, 513, 1025)])
def test_segment_counts(nprof, qlen):
    rng = np.random.default_rng(nprof)
    lens = rng.integers(30, 44, nprof)
    q = SynthDB.from_lengths(201, [qlen])
    d = SynthDB.from_lengths(202, lens)
    print(f"segments: {nprof} profiles, query {qlen}", flush=True)
    cbp = processing()
    cbp.TransferQueries(q)
    cbp.TransferCPMData(d)
    assert np.array_equal(cbp.phase1_keys(0), expected_keys(oracle(), q, 0, d))


@pytest.mark.parametrize("order", ["longest", "shortest", "mixed"])
def test_segment_order_and_batches(order):
    rng = np.random.default_rng(5)
    lens = np.sort(np.clip(np.rint(120 * np.exp(0.668 * rng.standard_normal(700))), 30, 900).astype(np.int32))
    lens = {"longest": lens[::-1], "shortest": lens, "mixed": rng.permutation(lens)}[order]
    q = SynthDB.from_lengths(211, [64, 65, 330])
    d = SynthDB.from_lengths(212, lens)
    d.plant(q, 213, 20, 3.0, 60.0)
    cbp = processing(dict(max_map_pairs=8))
    cbp.TransferQueries(q)
    cbp.TransferCPMData(d)
    cbp.SetDbDetails(d.npos, d.nprof)
    print(f"segment order {order}", flush=True)
    one = [cbp.ProcessScoreMatrix(i) for i in range(3)]
    for qs in ([0, 1, 2], [0, 2], [0, 1, 2] * 6):
        for i, r in zip(qs, cbp.ProcessBatch(qs)):
            assert np.array_equal(r["alndata"].view(np.uint32), one[i]["alndata"].view(np.uint32)), (order, qs, i)
            assert np.array_equal(r["order"], one[i]["order"])
            assert np.array_equal(r["aln_raw"], one[i]["aln_raw"])
    keys = cbp.phase1_keys(2)
    pick = np.linspace(0, d.nprof - 1, 40).astype(int)
    orc = oracle()
    from comer2_amd.host import encode_key
    for dp in pick:
        S, _ = orc.score_f32(q.view, 2, d.view, int(dp))
        m, _, _ = orc.viterbi_f32(q.view, 2, d.view, int(dp), S)
        assert int(keys[dp]) == encode_key(m.maxsc, m.x, m.y), (order, dp)


# 4 and 8 waves per workgroup over segments of several profiles (two or three,
# and about six), none of them long: 513-1,024 segments and more
@pytest.mark.parametrize("nprof,hi,waves", [(1700, 40, 4), (3600, 40, 8), (14000, 120, 8)])
@pytest.mark.parametrize("lq,rmax", [(60, 1), (100, 1), (120, 5), (200, 2), (180, 5), (340, 5), (250, 5), (500, 5), (310, 5)])
def test_segments_of_several_profiles(lq, rmax, nprof, hi, waves):
    rng = np.random.default_rng(nprof)
    lens = rng.integers(24, hi + 1, nprof)
    q = SynthDB.from_lengths(241, [lq])
    d = SynthDB.from_lengths(242, lens)
    print(f"segments of several: Lq={lq} rmax={rmax} nprof={nprof}", flush=True)
    cbp = processing()
    cbp.set_tuning(4096, rmax, 8)
    cbp.TransferQueries(q)
    cbp.TransferCPMData(d)
    keys = cbp.phase1_keys(0)
    assert cbp.last_phase1_shape() == (waves, False)
    orc = oracle()
    from comer2_amd.host import encode_key
    for dp in [int(i) for i in np.linspace(0, nprof - 1, 60)]:
        S, _ = orc.score_f32(q.view, 0, d.view, dp)
        m, _, _ = orc.viterbi_f32(q.view, 0, d.view, dp, S)
        assert int(keys[dp]) == encode_key(m.maxsc, m.x, m.y), (lq, rmax, dp, int(lens[dp]))
    cbp.set_tuning(4096, rmax, 1)
    assert np.array_equal(keys, cbp.phase1_keys(0))
    assert cbp.last_phase1_shape() == (1, False)


def test_more_batch_sizes_than_segment_sets_are_kept():
    """every size of batch cuts this chunk differently; eight sets are kept, and
    replayed batches meet sets made anew"""
    q = SynthDB.from_lengths(251, [60, 70])
    d = SynthDB.from_lengths(252, [200] * 1500)
    d.plant(q, 253, 8, 3.0, 60.0)
    cbp = processing(dict(max_map_pairs=8))
    cbp.TransferQueries(q)
    cbp.TransferCPMData(d)
    cbp.SetDbDetails(d.npos, d.nprof)
    one = [cbp.ProcessScoreMatrix(i) for i in range(2)]
    cbp.set_graph(True)
    for nq in list(range(4, 16)) + [4, 4, 4, 9, 9, 9, 4]:
        print(f"segment sets: batch of {nq}", flush=True)
        for i, r in enumerate(cbp.ProcessBatch([k % 2 for k in range(nq)])):
            assert np.array_equal(r["alndata"].view(np.uint32), one[i % 2]["alndata"].view(np.uint32)), (nq, i)
            assert np.array_equal(r["aln_raw"], one[i % 2]["aln_raw"]), (nq, i)
