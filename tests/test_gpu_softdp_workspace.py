"""Soft-DP calls that share one workspace from several streams, directly and
inside a captured graph: they follow each other, so each gives what it gives
alone."""
import numpy as np
import pytest
from comer2_amd._ffi import SynthDB
from gpu_common import processing

pytestmark = pytest.mark.gpu


def _prepared(n=12, ckpt=0):
    import torch
    from comer2_amd.softdp import SoftDP
    rng = np.random.default_rng(7)
    lens = rng.integers(600, 900, 2 * n).astype(np.int32)      # three to four bands a pair
    cbp = processing()
    cbp.TransferQueries(SynthDB.from_lengths(321, lens[:n]))
    cbp.TransferCPMData(SynthDB.from_lengths(322, lens[n:]))
    sdp = SoftDP(cbp, [(k, k) for k in range(n)], ckpt=ckpt)
    S = sdp.scores()
    th = torch.tensor([0.1, -0.2, 0.05, -0.1, 0.1], device="cuda")
    ins = [S, 0.5 * S, S - 0.25]
    ref = [sdp.forward(s, th) for s in ins]
    torch.cuda.synchronize()
    return cbp, sdp, ins, th, ref


def test_forwards_on_several_streams():
    import torch
    cbp, sdp, ins, th, ref = _prepared()
    streams = [torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.default_stream()]
    for rep in range(4):
        print(f"workspace: streams, pass {rep}", flush=True)
        got = []
        for k in range(6):
            with torch.cuda.stream(streams[k % 3]):
                got.append(sdp.forward(ins[(k + rep) % 3], th))
        torch.cuda.synchronize()
        for k in range(6):
            assert torch.equal(got[k], ref[(k + rep) % 3]), (rep, k)


@pytest.mark.parametrize("ckpt", [0, 32])
def test_step_and_next_forward_on_two_streams(ckpt):
    import torch
    cbp, sdp, ins, th, ref = _prepared(ckpt=ckpt)
    z = sdp.forward(ins[0], th)
    d0 = sdp.adjoint(ins[0], th, z)[0]
    torch.cuda.synchronize()
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    for rep in range(4):
        print(f"workspace: step and forward, ckpt {ckpt}, pass {rep}", flush=True)
        with torch.cuda.stream(s1):
            z1 = sdp.forward(ins[0], th)
            d1 = sdp.adjoint(ins[0], th, z1)[0]
        with torch.cuda.stream(s2):
            z2 = sdp.forward(ins[1], th)
        torch.cuda.synchronize()
        assert torch.equal(z1, ref[0]) and torch.equal(d1, d0) and torch.equal(z2, ref[1]), (ckpt, rep)


def test_captured_calls_on_two_streams():
    """two forked streams of one capture; replays with direct calls between"""
    import torch
    cbp, sdp, ins, th, ref = _prepared()
    main, side = torch.cuda.Stream(), torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    main.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(g, stream=main):
        side.wait_stream(main)
        a = sdp.forward(ins[0], th)
        with torch.cuda.stream(side):
            b = sdp.forward(ins[1], th)
        main.wait_stream(side)
        c = sdp.forward(ins[2], th)
    for rep in range(4):
        print(f"workspace: capture, replay {rep}", flush=True)
        for t in (a, b, c):
            t.zero_()
        e = sdp.forward(ins[rep % 3], th)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(e, ref[rep % 3]), rep
        for t, r in zip((a, b, c), ref):
            assert torch.equal(t, r), rep


@pytest.mark.parametrize("ckpt", [0, 32])
def test_workspace_at_any_float(ckpt):
    """a workspace that starts one, two or three floats into an allocation"""
    import torch
    cbp, sdp, ins, th, ref = _prepared(ckpt=ckpt)
    z = sdp.forward(ins[0], th)
    want = sdp.adjoint(ins[0], th, z, want_post=True)
    room = torch.empty(sdp.ws.numel() + 3, dtype=torch.float32, device="cuda")
    for off in (1, 2, 3):
        print(f"workspace: {4 * off} bytes in, ckpt {ckpt}", flush=True)
        sdp.ws = room[off:off + sdp.ws_bytes // 4]
        z2 = sdp.forward(ins[0], th)
        got = sdp.adjoint(ins[0], th, z2, want_post=True)
        torch.cuda.synchronize()
        assert torch.equal(z2, z) and all(torch.equal(x, y) for x, y in zip(got, want)), off
