"""Soft-DP score matrices against the oracle, bit for bit, at the edges of the
row items (32 rows, four at a time) and of the column blocks (64 columns per
wave, 256 per workgroup), with and without the secondary-structure term."""
import numpy as np
import pytest
from comer2_amd._ffi import SynthDB
from gpu_common import oracle, processing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ssswgt", [0.12, 0.0])
def test_score_matrices(ssswgt):
    import torch
    from comer2_amd.softdp import SoftDP
    rows = [1, 3, 4, 31, 32, 33, 37, 64, 130]
    cols = [1, 63, 64, 65, 255, 256, 257, 320, 2]
    q = SynthDB.from_lengths(321, rows)
    d = SynthDB.from_lengths(322, cols)
    opts = dict(ssswgt=ssswgt)
    cbp, orc = processing(opts), oracle(opts)
    cbp.TransferQueries(q)
    cbp.TransferCPMData(d)
    pairs = [(k, k) for k in range(len(rows))] + [(0, 6), (6, 0), (8, 5)]
    sdp = SoftDP(cbp, pairs, ckpt=0)
    S = sdp.scores()
    torch.cuda.synchronize()
    S = S.cpu().numpy()
    for (a, b), o, (L1, L2) in zip(sdp.pairs, sdp.offsets, sdp.shapes):
        exp = orc.score_f32(q.view, a, d.view, b)[0].ravel()
        assert np.array_equal(S[o:o + L1 * L2], exp), (ssswgt, L1, L2)
