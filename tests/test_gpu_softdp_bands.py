"""Soft-DP forward and adjoint against the FP64 oracle at the edges of the
stripes (64 rows), of the bands (4 stripes) that hand their rows over between
workgroups, of the groups of four columns and of the blocks of 64, with every
cell stored and with each checkpoint interval.  Tolerances: log Z 1e-5
relative, gradients and posteriors 1e-4 absolute (they lie in [0, 1]), the
offsets' gradients 1e-3 relative, as for the other soft-DP tests."""
import numpy as np
import pytest
from comer2_amd._ffi import SynthDB
from gpu_common import oracle, processing

pytestmark = pytest.mark.gpu

ROWS = [1, 2, 63, 64, 65, 128, 255, 256, 257, 320, 513, 300]
COLS = [1, 130, 3, 64, 65, 1, 66, 4, 63, 129, 62, 300]


@pytest.mark.parametrize("ckpt", [0, 16, 32, 64])
def test_band_edges(ckpt):
    import torch
    from comer2_amd.softdp import SoftDP
    q = SynthDB.from_lengths(331, ROWS)
    d = SynthDB.from_lengths(332, COLS)
    d.plant(q, 333, 6, 20.0, 60.0)
    cbp = processing()
    cbp.TransferQueries(q)
    cbp.TransferCPMData(d)
    orc = oracle()
    pairs = [(k, k) for k in range(len(ROWS))] + [(10, 11), (0, 11), (8, 0), (7, 7)]
    sdp = SoftDP(cbp, pairs, ckpt=ckpt)
    Sh = np.concatenate([orc.score_f32(q.view, a, d.view, b)[0].ravel() for a, b in sdp.pairs]).astype(np.float32)
    S = torch.from_numpy(Sh).cuda()
    th = torch.tensor([0.1, -0.2, 0.05, -0.1, 0.1], dtype=torch.float32, device="cuda")
    w = torch.linspace(0.5, 1.5, len(pairs), device="cuda")
    for rep in range(2):
        print(f"soft dp bands: ckpt {ckpt}, pass {rep}", flush=True)
        logZ = sdp.forward(S, th)
        dS, dth, post = sdp.adjoint(S, th, logZ, w, want_post=True)
        torch.cuda.synchronize()
        z, g, t, p, wn = (x.cpu().numpy() for x in (logZ, dS, dth, post, w))
        thd = th.cpu().numpy().astype(np.float64)
        for k, (a, b) in enumerate(sdp.pairs):
            L1, L2 = sdp.shapes[k]
            o = int(sdp.offsets[k])
            ez, eS, eth, ep = orc.sdp_grad(q.view, a, d.view, b, Sh[o:o + L1 * L2].reshape(L1, L2).astype(np.float64), thd)
            ctx = (ckpt, rep, L1, L2)
            assert abs(z[k] - ez) <= 1e-5 * abs(ez), ctx
            assert np.max(np.abs(g[o:o + L1 * L2] - wn[k] * eS.ravel())) < 1e-4, ctx
            assert np.max(np.abs(p[o:o + L1 * L2] - ep.ravel())) < 1e-4, ctx
            assert np.all(np.abs(t[k] - wn[k] * eth) <= 1e-3 * np.maximum(1.0, np.abs(eth))), (ctx, t[k], eth)
