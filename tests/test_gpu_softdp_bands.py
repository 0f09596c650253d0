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


def _check(orc, q, d, sdp, Sh, thd, got, ks, ctx):
    """log Z, gradients, posteriors and offset gradients of pairs ks against
    the oracle, at the tolerances above"""
    z, g, t, p = got
    for k in ks:
        a, b = sdp.pairs[k]
        L1, L2 = sdp.shapes[k]
        o = int(sdp.offsets[k])
        ez, eS, eth, ep = orc.sdp_grad(q.view, a, d.view, b, Sh[o:o + L1 * L2].reshape(L1, L2).astype(np.float64), thd)
        c = ctx + (k, L1, L2)
        assert abs(z[k] - ez) <= 1e-5 * abs(ez), c
        assert np.max(np.abs(g[o:o + L1 * L2] - eS.ravel())) < 1e-4, c
        assert np.max(np.abs(p[o:o + L1 * L2] - ep.ravel())) < 1e-4, c
        assert np.all(np.abs(t[k] - eth) <= 1e-3 * np.maximum(1.0, np.abs(eth))), (c, t[k], eth)


def _step(sdp, S, th):
    import torch
    logZ = sdp.forward(S, th)
    dS, dth, post = sdp.adjoint(S, th, logZ, want_post=True)
    torch.cuda.synchronize()
    return [x.cpu().numpy() for x in (logZ, dS, dth, post)]


# 1,280 bands of two to a pair for at most 1,024 workgroups, and 4,500 pairs of
# one stripe each for 4,096: workgroups take a second and third item
@pytest.mark.parametrize("ckpt", [0, 64])
@pytest.mark.parametrize("npairs,rows,cols", [(640, (257, 300), (20, 40)), (4500, (1, 64), (1, 40))])
def test_more_items_than_workgroups(npairs, rows, cols, ckpt):
    import torch
    from comer2_amd.softdp import SoftDP
    rng = np.random.default_rng(npairs)
    n = 50
    q = SynthDB.from_lengths(341, rng.integers(rows[0], rows[1] + 1, n).astype(np.int32))
    d = SynthDB.from_lengths(342, rng.integers(cols[0], cols[1] + 1, n).astype(np.int32))
    cbp = processing()
    cbp.TransferQueries(q)
    cbp.TransferCPMData(d)
    orc = oracle()
    sdp = SoftDP(cbp, [(k % n, k % n) for k in range(npairs)], ckpt=ckpt)
    print(f"soft dp items: {npairs} pairs of {rows} rows, ckpt {ckpt}", flush=True)
    one = [orc.score_f32(q.view, k, d.view, k)[0].ravel() for k in range(n)]
    Sh = np.concatenate([one[k % n] for k in range(npairs)]).astype(np.float32)
    th = torch.tensor([0.1, -0.2, 0.05, -0.1, 0.1], dtype=torch.float32, device="cuda")
    z, g, t, p = got = _step(sdp, torch.from_numpy(Sh).cuda(), th)
    for k in range(n, npairs):
        a, b, m = int(sdp.offsets[k]), int(sdp.offsets[k % n]), one[k % n].size
        assert z[k] == z[k % n] and np.array_equal(t[k], t[k % n]), k
        assert np.array_equal(g[a:a + m], g[b:b + m]) and np.array_equal(p[a:a + m], p[b:b + m]), k
    _check(orc, q, d, sdp, Sh, th.cpu().numpy().astype(np.float64), got, range(0, n, 3), (npairs, ckpt))


# cells that must not match: their terms are zero in log Z and every gradient
@pytest.mark.parametrize("mask", [-np.inf, np.finfo(np.float32).min, -1e30])
@pytest.mark.parametrize("ckpt", [0, 32])
def test_masked_scores(mask, ckpt):
    import torch
    from comer2_amd.softdp import SoftDP
    rows, cols = [70, 300, 1, 64, 130], [90, 65, 40, 1, 300]
    q = SynthDB.from_lengths(351, rows)
    d = SynthDB.from_lengths(352, cols)
    d.plant(q, 353, 4, 20.0, 60.0)
    cbp = processing()
    cbp.TransferQueries(q)
    cbp.TransferCPMData(d)
    orc = oracle()
    pairs = [(k, k) for k in range(5)] + [(1, 4), (0, 0)]
    sdp = SoftDP(cbp, pairs, ckpt=ckpt)
    rng = np.random.default_rng(9)
    blocks = []
    for k, (a, b) in enumerate(sdp.pairs):
        s = orc.score_f32(q.view, a, d.view, b)[0].astype(np.float32).copy()
        s[rng.random(s.shape) < 0.2] = mask
        s[rng.integers(0, s.shape[0], 3)] = mask                 # whole rows and columns
        s[:, rng.integers(0, s.shape[1], 3)] = mask
        if k == 5:
            s[:, 0] = s[0] = s[-1] = s[:, -1] = mask             # the matrix's edges
        if k == 6:
            s[:] = mask                                          # everything
        blocks.append(s.ravel())
    Sh = np.concatenate(blocks)
    print(f"soft dp masked: {mask}, ckpt {ckpt}", flush=True)
    th = torch.tensor([0.1, -0.2, 0.05, -0.1, 0.1], dtype=torch.float32, device="cuda")
    got = _step(sdp, torch.from_numpy(Sh).cuda(), th)
    assert all(np.isfinite(x).all() for x in got)
    _check(orc, q, d, sdp, Sh, th.cpu().numpy().astype(np.float64), got, range(len(pairs)), (mask, ckpt))
    o = int(sdp.offsets[6])
    assert np.max(np.abs(got[1][o:])) < 1e-4 and abs(got[0][6] - np.log(70 * 90)) < 1e-4


@pytest.mark.parametrize("ckpt", [0, 32])
def test_not_a_number_stays_in_its_pair(ckpt):
    """scores that are not numbers, among them the bit pattern by which bands
    wait for each other's rows: their pair's results are none, every wait ends
    and the other pairs' results are what they are without"""
    import torch
    from comer2_amd.softdp import SoftDP
    q = SynthDB.from_lengths(361, [300, 520, 64])
    d = SynthDB.from_lengths(362, [150, 260, 70])
    cbp = processing()
    cbp.TransferQueries(q)
    cbp.TransferCPMData(d)
    sdp = SoftDP(cbp, [(0, 0), (1, 1), (2, 2), (0, 1)], ckpt=ckpt)
    S = sdp.scores()
    th = torch.zeros(5, dtype=torch.float32, device="cuda")
    ref = _step(sdp, S, th)
    o, n = int(sdp.offsets[1]), 520 * 260
    for bits in (-1, 0x7FC00000, 0x7F800000):
        print(f"soft dp not a number: {bits & 0xFFFFFFFF:08x}, ckpt {ckpt}", flush=True)
        bad = S.clone()
        bad[o:o + n].view(torch.int32).view(520, 260)[200:260, 40:200] = bits
        z, g, t, p = _step(sdp, bad, th)
        assert not np.isfinite(z[1])
        for k in (0, 2, 3):
            a, m = int(sdp.offsets[k]), sdp.shapes[k][0] * sdp.shapes[k][1]
            assert z[k] == ref[0][k] and np.array_equal(t[k], ref[2][k]), (bits, k)
            assert np.array_equal(g[a:a + m], ref[1][a:a + m]) and np.array_equal(p[a:a + m], ref[3][a:a + m])
