"""Soft-DP calls of two handles on torch's default stream: a result that is
dropped hands its memory to the next call at once, so the calls must run in
the order they were made."""
import numpy as np
import pytest
from comer2_amd._ffi import SynthDB
from gpu_common import processing

pytestmark = pytest.mark.gpu


def _pairs(seed, n):
    from comer2_amd.softdp import SoftDP
    lens = np.full(n, 300)
    cbp = processing()
    cbp.TransferQueries(SynthDB.from_lengths(seed, lens))
    cbp.TransferCPMData(SynthDB.from_lengths(seed + 1, lens))
    return cbp, SoftDP(cbp, [(k, k) for k in range(n)], ckpt=0)


def test_two_handles_on_the_default_stream():
    import torch
    (ca, a), (cb, b) = _pairs(301, 24), _pairs(311, 24)
    th = torch.zeros(5, device="cuda")
    ref = a.scores()
    z = a.forward(ref, th)
    dS = a.adjoint(ref, th, z)[0]
    torch.cuda.synchronize()
    for _ in range(20):
        b.scores()                       # dropped: the next call's block
        s = a.scores()
        b.forward(ref, th)
        z2 = a.forward(s, th)
        d2 = a.adjoint(s, th, z2)[0]
        torch.cuda.synchronize()
        assert torch.equal(s, ref) and torch.equal(z2, z) and torch.equal(d2, dS)
