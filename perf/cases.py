"""Timed workloads of the search path and of the differentiable soft DP.

Every case is one call sequence that a program using this framework makes on
the GPU, through the public entry points:

- ``search``   one query against the uploaded database chunk
               (``CuBatchProcessing.ProcessScoreMatrix``): score, Viterbi,
               statistics, realignment or drawing, records and strings;
- ``batch``    several queries against the chunk in one call (``ProcessBatch``);
- ``stream``   a database in host memory, uploaded in chunks while the chunk
               before is searched (``SearchDB``);
- ``keys``     the phase-1 maxima of every profile alone (``phase1_keys``);
- ``scores``   score matrices of (query, profile) pairs (``SoftDP.scores``);
- ``softdp``   a training step: log Z of the pairs and the gradients of a
               weighted sum for the scores and the five gap offsets, through
               the torch binding (``soft_dp`` and ``torch.autograd.grad``);
- ``posterior`` log Z, gradients and match posteriors by the explicit calls
               (``SoftDP.forward``, ``SoftDP.adjoint``).

Inputs come from the seeded generator with the length distributions and the
planted homologs of the benchmark.  Everything is FP32, the only type of the
path; the options that change the computation (MAPALN, the context-vector
weight, checkpointing) each have a case.
"""
import math

import numpy as np
import torch

from comer2_amd._ffi import SynthDB
from comer2_amd.host import CuBatchProcessing
from comer2_amd.softdp import SoftDP, soft_dp

SIGMA = 0.668                       # of the log-normal profile lengths
KMIN, KMAX = 3.0, 60.0              # concentrations of the planted homologs


def listed():
    return [
        # a few profiles, as an interactive check of one family: latency
        dict(name="search_tiny", kind="search", qlen=87, nprof=150, median=120, maxlen=800,
             nplant=6, cap=0, mapaln=1, cv=0),
        # the small benchmark configuration: 150 positions, 2,000 profiles, best 100 realigned
        dict(name="search_small", kind="search", qlen=150, nprof=2000, median=180, maxlen=800,
             nplant=40, cap=100, mapaln=1, cv=0),
        # the headline search (one query of 300 positions, planted homologs, best 2,000
        # realigned) against a database of a third of its size
        dict(name="search_large", kind="search", qlen=300, nprof=60000, median=200, maxlen=3000,
             nplant=1200, cap=2000, mapaln=1, cv=0),
        # a multi-domain query: several stripes of rows, long realignments
        dict(name="search_long_query", kind="search", qlen=1337, nprof=12000, median=200, maxlen=3000,
             nplant=200, cap=200, mapaln=1, cv=0),
        # alignments drawn from the phase-1 path (MAPALN = 0)
        dict(name="search_viterbi", kind="search", qlen=223, nprof=15000, median=200, maxlen=3000,
             nplant=400, cap=0, mapaln=0, cv=0),
        # profiles with context vectors, scored with the shipped option file's weight
        dict(name="search_context", kind="search", qlen=181, nprof=6000, median=200, maxlen=2000,
             nplant=120, cap=100, mapaln=1, cv=1),
        # a batch of queries of mixed lengths, the serving shape
        dict(name="batch_queries", kind="batch", nq=24, qmin=50, qmax=1000, nprof=15000, median=200,
             maxlen=3000, nplant=480, cap=100),
        # a database larger than the device's share, in host memory
        dict(name="stream_database", kind="stream", qlen=257, nprof=12000, median=200, maxlen=3000,
             nplant=200, cap=200, chunk=800000),
        # the prefilter alone, a domain-sized query
        dict(name="keys_short_query", kind="keys", qlen=61, nprof=30000, median=200, maxlen=3000),
        # score matrices of a training batch
        dict(name="softdp_scores", kind="scores", npairs=1024, lmin=50, lmax=600),
        # a training step on a batch of single-domain pairs, every forward cell kept
        dict(name="softdp_step", kind="softdp", npairs=1024, lmin=50, lmax=600, ckpt=0),
        # long pairs at the automatic checkpoint interval, with posteriors
        dict(name="softdp_long", kind="posterior", npairs=24, lmin=2000, lmax=5000, ckpt=-1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["search", "search", "search", "batch", "stream", "keys", "scores", "softdp", "posterior"])
    if kind == "search":
        qlen = _log(rng, 40, 1400)
        cv = int(rng.random() < 0.2)
        nprof = _log(rng, 100, min(60000, 6000 if cv else 18000000 // qlen))
        return dict(kind=kind, qlen=qlen, nprof=nprof, median=rng.randint(100, 220), maxlen=rng.choice([800, 2000, 3000]),
                    nplant=max(2, nprof // rng.randint(40, 100)), cap=rng.choice([0, 100, 2000]),
                    mapaln=int(rng.random() < 0.75), cv=cv)
    if kind == "batch":
        nprof = _log(rng, 200, 15000)
        nq = rng.randint(2, 24)
        return dict(kind=kind, nq=nq, qmin=50, qmax=rng.randint(200, 1000), nprof=nprof, median=rng.randint(120, 200),
                    maxlen=rng.choice([800, 3000]), nplant=max(nq, nprof // 40), cap=100)
    if kind == "stream":
        nprof = _log(rng, 1000, 12000)
        return dict(kind=kind, qlen=_log(rng, 60, 600), nprof=nprof, median=200, maxlen=3000,
                    nplant=nprof // 60, cap=200, chunk=max(50000, nprof * 250 // rng.randint(2, 5)))
    if kind == "keys":
        qlen = _log(rng, 30, 900)
        return dict(kind=kind, qlen=qlen, nprof=_log(rng, 100, min(30000, 9000000 // qlen)),
                    median=rng.randint(100, 220), maxlen=rng.choice([800, 3000]))
    if kind in ("scores", "softdp"):
        lmax = _log(rng, 64, 700)
        c = dict(kind=kind, npairs=_log(rng, 4, min(1024, 90000000 // (lmax * lmax))), lmin=max(20, lmax // rng.randint(2, 12)),
                 lmax=lmax)
        if kind == "softdp":
            c["ckpt"] = rng.choice([0, 0, -1])
        return c
    lmax = _log(rng, 700, 5000)
    return dict(kind=kind, npairs=_log(rng, 2, 24), lmin=lmax * 2 // 5, lmax=lmax, ckpt=rng.choice([-1, -1, 0]))


# --------------------------------------------------------------------------
# inputs

def _lengths(case, n, lo, hi, median=0):
    """n profile lengths of the case, the same for every seed: log-normal around
    the median and longest first, as a database is stored, or uniform"""
    rng = np.random.default_rng([n, lo, hi, int(median), case.get("qlen", 0)])
    if median:
        x = np.rint(median * np.exp(SIGMA * rng.standard_normal(n)))
        return np.sort(np.clip(x, lo, hi).astype(np.int32))[::-1]
    return rng.integers(lo, hi + 1, n).astype(np.int32)


def _search_sets(case, seed):
    """query set and database with planted homologs"""
    base = 1000003 * seed
    if case["kind"] == "batch":
        q = SynthDB.from_lengths(base + 1, _lengths(case, case["nq"], case["qmin"], case["qmax"]))
    else:
        q = SynthDB.from_lengths(base + 1, [case["qlen"]])
    d = SynthDB.from_lengths(base + 2, _lengths(case, case["nprof"], 30, case["maxlen"], case["median"]))
    if case.get("cv"):
        q.add_cv(base + 3)
        d.add_cv(base + 4)
    if case.get("nplant"):
        d.plant(q, base + 5, case["nplant"], KMIN, KMAX)
    return q, d


def _pair_sets(case, seed):
    base = 1000003 * seed
    n = case["npairs"]
    lens = _lengths(case, 2 * n, case["lmin"], case["lmax"])
    return SynthDB.from_lengths(base + 1, lens[:n]), SynthDB.from_lengths(base + 2, lens[n:])


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _field(view, name, shape):
    return np.ctypeslib.as_array(getattr(view, name), shape)


def _scores64(q, d):
    """score matrices of the pairs (k, k) in 64 bits, packed one after another:
    log(sum_a q_a d_a / (0.5 (bq_a + bd_a))) - 0.002 + 0.12 x the
    secondary-structure term"""
    from comer2_amd import tables
    dev = _device()
    tab = torch.from_numpy(tables.load_ssss().reshape(30, 30)).to(dev).double()
    sides = []
    for s in (q, d):
        v, npos = s.view, s.npos
        trg = torch.from_numpy(_field(v, "trgfrq", (20, npos)).copy()).to(dev).double()
        ssp = torch.from_numpy(_field(v, "ssprb", (3, npos)).copy()).to(dev)
        bins = (ssp * 9.999).int().long()                   # FP32 product, as the bins are defined
        onehot = torch.zeros((30, npos), dtype=torch.float64, device=dev)
        for j in range(3):
            onehot.scatter_(0, (bins[j] + 10 * j)[None], ssp[j].double()[None])
        bkg = torch.from_numpy(_field(v, "bkg", (20, s.nprof)).copy()).to(dev).double()
        sides.append((trg, onehot, ssp[2].double() + 0.1, bkg, s.dists(), s.lengths()))
    out = []
    for k in range(q.nprof):
        (tq, oq, hq, bq), (q0, l1) = sides[0][:4], (int(sides[0][4][k]), int(sides[0][5][k]))
        (td, od, hd, bd), (d0, l2) = sides[1][:4], (int(sides[1][4][k]), int(sides[1][5][k]))
        w = 2.0 / (bq[:, k] + bd[:, k])
        a = tq[:, q0:q0 + l1]
        s = torch.log(a.T @ (td[:, d0:d0 + l2] * w[:, None])) - 0.002
        ss = oq[:, q0:q0 + l1].T @ (tab @ od[:, d0:d0 + l2])
        ss = ss + hq[q0:q0 + l1, None] * hd[None, d0:d0 + l2] * 0.1111111 - 0.05
        out.append((s + 0.12 * ss).reshape(-1))
    return torch.cat(out)


def _pair_inputs(case, seed, q, d):
    """scores of the pairs, gap offsets and the weights of the step's loss"""
    rng = np.random.default_rng(seed)
    S = _scores64(q, d).float()
    theta = torch.tensor(rng.uniform(-0.2, 0.2, 5), dtype=torch.float32, device=S.device)
    w = torch.tensor(rng.uniform(0.5, 1.5, case["npairs"]), dtype=torch.float32, device=S.device)
    return S, theta, w


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("scores", "softdp", "posterior"):
        q, d = _pair_sets(case, seed)
        cbp = CuBatchProcessing(0)
        cbp.TransferQueries(q)
        cbp.TransferCPMData(d)
        sdp = SoftDP(cbp, [(k, k) for k in range(case["npairs"])], ckpt=case.get("ckpt", 0))
        st = dict(kind=kind, q=q, d=d, cbp=cbp, sdp=sdp)
        if kind != "scores":
            st["S"], st["theta"], st["w"] = _pair_inputs(case, seed, q, d)
        if kind == "softdp":
            st["S"].requires_grad_(True)
            st["theta"].requires_grad_(True)
        return st
    q, d = _search_sets(case, seed)
    opts = dict(max_map_pairs=case.get("cap", 0), mapaln=case.get("mapaln", 1))
    if case.get("cv"):
        opts["cvswgt"] = 0.15
    cbp = CuBatchProcessing(0, options=opts)
    cbp.TransferQueries(q)
    if kind != "stream":
        cbp.TransferCPMData(d)
    cbp.SetDbDetails(d.npos, d.nprof)
    rows = 2 * case.get("nplant", 0) // (q.nprof if q.nprof < 8 else q.nprof // 4) + 64
    return dict(kind=kind, q=q, d=d, cbp=cbp, nq=q.nprof, chunk=case.get("chunk", 0), rows=rows,
                width=int(q.lengths().max()) + int(d.lengths().max()) + 64)


_RECORD = ("score", "pronr", "dst", "psts", "beg", "end", "logE", "epa", "lmbd", "K", "H", "E", "smin", "smax",
           "lmbdest", "kest", "idnts", "ngaps", "alnlen", "order", "map_rows")


def _records(state, results):
    """the queries' whole results in arrays that hold a fixed number of hits: the
    hits' records, their order, the rows realigned and their strings"""
    n, rows = len(results), state["rows"]
    out = {k: np.zeros((n, rows), results[0][k].dtype) for k in _RECORD}
    out["strings"] = np.zeros((n, rows, 3, state["width"]), np.uint8)
    out["counts"] = np.array([[r["npassed"], r["nposits"], r["maxlen"], r["nmap"]] for r in results], np.int64)
    out["limits"] = np.array([[r["scorethld"], r["logevthld"], r["search_space"]] for r in results], np.float64)
    for i, r in enumerate(results):
        for k in _RECORD:
            x = r[k]
            out[k][i, :x.size] = x
        raw = r["aln_raw"]
        out["strings"][i, :raw.shape[0], :, :raw.shape[2]] = raw
    return out


def run(state):
    kind, cbp = state["kind"], state["cbp"]
    if kind == "search":
        return _records(state, [cbp.ProcessScoreMatrix(0)])
    if kind == "batch":
        return _records(state, cbp.ProcessBatch(list(range(state["nq"]))))
    if kind == "stream":
        return _records(state, cbp.SearchDB(state["d"], [0], chunk_pos=state["chunk"]))
    if kind == "keys":
        return cbp.phase1_keys(0)
    sdp = state["sdp"]
    if kind == "scores":
        return sdp.scores()
    if kind == "softdp":
        logZ = soft_dp(state["S"], state["theta"], sdp)
        dS, dtheta = torch.autograd.grad((logZ * state["w"]).sum(), (state["S"], state["theta"]))
        return {"logZ": logZ.detach(), "dS": dS, "dtheta": dtheta}
    logZ = sdp.forward(state["S"], state["theta"])
    dS, dtheta, post = sdp.adjoint(state["S"], state["theta"], logZ, state["w"], want_post=True)
    return {"logZ": logZ, "dS": dS, "dtheta": dtheta, "post": post}


def work(case):
    """operations and bytes of one pass: per search cell 41 for the score, 10 for
    the secondary-structure term, 36 for the five-state recurrence (context
    vectors: 45 more), the database's fields read once; per soft-DP cell 83
    forward and 130 in the adjoint (a transcendental counted as one), the
    scores read once and the outputs written once"""
    kind = case["kind"]
    if kind in ("scores", "softdp", "posterior"):
        mean = 0.5 * (case["lmin"] + case["lmax"])
        cells = case["npairs"] * mean * mean
        if kind == "scores":
            return {"bytes": 4 * cells + 2 * 92 * case["npairs"] * mean, "flops": 51 * cells}
        return {"bytes": (12 if kind == "posterior" else 8) * cells, "flops": 213 * cells}
    rows = case["nq"] * 0.5 * (case["qmin"] + case["qmax"]) if kind == "batch" else case["qlen"]
    npos = case["nprof"] * min(case["median"] * math.exp(0.5 * SIGMA * SIGMA), case["maxlen"])
    flops = 87 + (45 if case.get("cv") else 0)
    return {"bytes": npos * (4 * 30 + (84 if case.get("cv") else 0)) + 8 * case["nprof"], "flops": flops * rows * npos}


# --------------------------------------------------------------------------
# the soft DP in 64 bits

def _lse(*x):
    m = x[0]
    for y in x[1:]:
        m = torch.maximum(m, y)
    s = torch.zeros_like(m)
    for y in x:
        s = s + torch.exp(y - m)
    return m + torch.log(s)


def _trans(s, rows):
    """[7][pairs][rows] transitions of the row classes at i (MI and II at i + 1), zero beyond a profile"""
    npos, n = s.npos, s.nprof
    t = _field(s.view, "trans", (7, npos + n)).astype(np.float64)
    out = np.zeros((7, n, rows))
    dist, length = s.dists(), s.lengths()
    for p in range(n):
        b, l = int(dist[p]) + p, int(length[p])
        for k in range(7):
            o = b + (1 if k in (1, 4) else 0)
            out[k, p, :l] = t[k, o:o + l]
    return torch.from_numpy(out).to(_device())


def _boundary(qt):
    """the vectors left of column 0 that the rows (left) and the diagonals (diag)
    see: each block of 32 rows swept over the 32 columns before the profile
    with transitions and scores of -99, from (0, -99, -99, -99, -99); rows 31 of
    a block see the initial values, and rows 0 and 31 on their diagonal"""
    n, rows = qt.shape[1], qt.shape[2]
    nb = (rows + 31) // 32
    q = torch.zeros((7, n, nb * 32), dtype=torch.float64, device=qt.device)
    q[:, :, :rows] = qt
    q = q.reshape(7, n, nb, 32)
    init = [torch.full((n, nb), v, dtype=torch.float64, device=qt.device) for v in (0.0, -99.0, -99.0, -99.0, -99.0)]

    def mexp(x):
        return torch.where(x > -16.0, torch.exp(x), torch.zeros_like(x))

    def mlog(x):
        return torch.where(x > 3.8e-11, torch.log(x.clamp_min(1e-300)), torch.full_like(x, -99.0))

    def lse2(a, b):
        m = torch.maximum(a, b)
        return mlog(mexp(a - m) + mexp(b - m)) + m

    prev = {}
    left = torch.empty((5, n, nb, 32), dtype=torch.float64, device=qt.device)
    diag = torch.empty_like(left)
    for r in range(32):
        t = [q[k, :, :, r] for k in range(7)]
        first, row, lf = 31 - r, {}, init
        for c in range(first, 32):
            up = prev.get(c, init) if c > first else init
            dg = prev.get(c - 1, init) if c - 1 > first else init
            a = [dg[1] + t[0] - 198, dg[2] + t[3] - 198, dg[3] + t[5] - 198, dg[4] + t[0] - 198, dg[0] + t[0] - 198]
            m = torch.zeros_like(a[0])
            for x in a:
                m = torch.maximum(m, x)
            s = mexp(-m)
            for x in a:
                s = s + mexp(x - m)
            lf = [mlog(s) + m, lse2(up[0] + t[0] - 99, up[1] + t[0] - 99), lse2(lf[0] + t[1] - 99, lf[2] + t[4] - 99),
                  lse2(up[0] + t[2], up[3] + t[6]), lse2(lf[0] - 99, lf[4] - 99)]
            row[c] = lf
        for k in range(5):
            left[k, :, :, r] = init[k] if r == 31 else row[31][k]
            diag[k, :, :, r] = init[k] if r in (0, 31) else prev[31][k]
        prev = row
    return left.reshape(5, n, nb * 32)[:, :, :rows], diag.reshape(5, n, nb * 32)[:, :, :rows]


def _softdp64(q, d, S, theta):
    """log Z, dlogZ/dS (packed), dlogZ/dtheta per pair and match posteriors
    (packed) in 64 bits, all pairs along their anti-diagonals at once"""
    dev = _device()
    L1 = torch.from_numpy(q.lengths().astype(np.int64)).to(dev)
    L2 = torch.from_numpy(d.lengths().astype(np.int64)).to(dev)
    n, m1, m2 = q.nprof, int(L1.max()), int(L2.max())
    th = [float(x) for x in theta.double().cpu()]
    qt = _trans(q, m1 + 1)                              # row m1: beyond every query
    left, diag = _boundary(qt[:, :, :m1])
    # column c of row i on anti-diagonal t is t - i: the profile reversed, so a slice is a diagonal
    W = m1 + 2
    dt = _trans(d, m2)
    rev = torch.zeros((7, n, m2 + 2 * W), dtype=torch.float64, device=dev)
    rev[:, :, W:W + m2] = dt.flip(2)

    def dcol(k, t, shift=0, rows=m1):                   # class k at column t + shift - i
        j = W + m2 - 1 - (t + shift)
        return rev[k, :, j:j + rows]

    # scores padded by W columns on both sides and a row below
    wid = m2 + 2 * W
    SP = torch.zeros((n, m1 + 1, wid), dtype=torch.float32, device=dev)
    o, l1, l2 = 0, L1.tolist(), L2.tolist()
    for p in range(n):
        SP[p, :l1[p], W:W + l2[p]] = S[o:o + l1[p] * l2[p]].reshape(l1[p], l2[p])
        o += l1[p] * l2[p]
    OUT = torch.zeros((n, m1 + 1, wid), dtype=torch.float64, device=dev)
    POST = torch.zeros_like(OUT)

    def sdiag(M, t, row=0):                             # M[p, i + row, t - i]
        return torch.as_strided(M, (n, m1), (M.stride(0), wid - 1), row * wid + W + t)

    rows = torch.arange(m1, device=dev)
    NEG = -1.0e30
    neg = torch.full((n, m1), NEG, dtype=torch.float64, device=dev)

    def down(x, top):                                   # value of row i - 1
        return torch.cat([torch.full((n, 1), top, dtype=torch.float64, device=dev), x[:, :-1]], 1)

    def below(x):                                       # value of row i + 1
        return torch.cat([x[:, 1:], torch.full((n, 1), NEG, dtype=torch.float64, device=dev)], 1)

    q0 = [qt[k, :, :m1] for k in range(7)]
    q1 = [qt[k, :, 1:m1 + 1] for k in range(7)]
    tops = (0.0, -99.0, -99.0, -99.0, -99.0)

    def near(t, F1, F2):
        """up, diagonal and left neighbours of anti-diagonal t"""
        c0 = rows[None] == t
        up = [down(F1[k], tops[k]) for k in range(5)]
        dg = [torch.where(c0, diag[k], down(F2[k], tops[k])) for k in range(5)]
        lf = [torch.where(c0, left[k], F1[k]) for k in range(5)]
        return up, dg, lf

    def terms(t, up, dg, lf):
        D = [dcol(k, t) for k in range(7)]
        s = sdiag(SP, t).double()
        a = (dg[1] + q0[0] + D[3] + th[4] + s, dg[2] + q0[3] + D[0] + th[4] + s, dg[3] + q0[5] + D[0] + th[4] + s,
             dg[4] + q0[0] + D[5] + th[4] + s, dg[0] + q0[0] + D[0] + s)
        return (a, (up[0] + q0[0] + D[1] + th[0], up[1] + q0[0] + D[4] + th[1]),
                (lf[0] + q0[1] + D[0] + th[0], lf[2] + q0[4] + D[0] + th[1]),
                (up[0] + q0[2] + th[2], up[3] + q0[6] + th[3]), (lf[0] + D[2] + th[2], lf[4] + D[6] + th[3]))

    nd = m1 + m2 - 1
    F = [None] * nd
    zm = torch.zeros((n,), dtype=torch.float64, device=dev)
    zs = torch.zeros_like(zm)
    F1 = F2 = [neg] * 5
    for t in range(nd):
        valid = (rows[None] < L1[:, None]) & (t - rows[None] >= 0) & (t - rows[None] < L2[:, None])
        a, b, c, e, g = terms(t, *near(t, F1, F2))
        cur = [_lse(*a, torch.zeros_like(a[0])), _lse(*b), _lse(*c), _lse(*e), _lse(*g)]
        cur = [torch.where(valid, x, neg) for x in cur]
        top = torch.maximum(zm, cur[0].max(1).values)
        zs = zs * torch.exp(zm - top) + torch.exp(cur[0] - top[:, None]).sum(1)
        zm = top
        F[t] = torch.stack(cur)
        F2, F1 = F1, F[t]
    Z = zm + torch.log(zs)
    dth = torch.zeros((n, 5), dtype=torch.float64, device=dev)
    B1 = B2 = [neg] * 5
    zero = torch.zeros_like(neg)
    for t in range(nd - 1, -1, -1):
        valid = (rows[None] < L1[:, None]) & (t - rows[None] >= 0) & (t - rows[None] < L2[:, None])
        D0 = [dcol(k, t) for k in range(7)]
        D1 = [dcol(k, t, 1) for k in range(7)]
        dg = below(B2[0]) + torch.as_strided(SP, (n, m1), (SP.stride(0), wid - 1), wid + W + t + 1).double()
        mi, dn, im, nd_ = below(B1[1]), below(B1[3]), B1[2], B1[4]
        cur = [_lse(zero, dg + q1[0] + D1[0], mi + q1[0] + D0[1] + th[0], im + q0[1] + D1[0] + th[0],
                    dn + q1[2] + th[2], nd_ + D1[2] + th[2]),
               _lse(dg + q1[0] + D1[3] + th[4], mi + q1[0] + D0[4] + th[1]),
               _lse(dg + q1[3] + D1[0] + th[4], im + q0[4] + D1[0] + th[1]),
               _lse(dg + q1[5] + D1[0] + th[4], dn + q1[6] + th[3]),
               _lse(dg + q1[0] + D1[5] + th[4], nd_ + D1[6] + th[3])]
        cur = [torch.where(valid, x, neg) for x in cur]
        f = F[t][0]
        bz = torch.where(valid, cur[0] - Z[:, None], neg)
        torch.as_strided(OUT, (n, m1), (OUT.stride(0), wid - 1), W + t).add_(
            torch.where(valid, torch.exp(bz) * torch.expm1(f.clamp_min(0.0)), zero))
        torch.as_strided(POST, (n, m1), (POST.stride(0), wid - 1), W + t).add_(
            torch.where(valid, torch.exp(bz + f), zero))
        a, b, c, e, g = terms(t, *near(t, F[t - 1] if t >= 1 else [neg] * 5, F[t - 2] if t >= 2 else [neg] * 5))
        w = [torch.where(valid, cur[k] - Z[:, None], neg) for k in range(5)]

        def cnt(x, k):
            return torch.exp(torch.where(valid, x + w[k], neg)).sum(1)
        dth[:, 4] += cnt(a[0], 0) + cnt(a[1], 0) + cnt(a[2], 0) + cnt(a[3], 0)
        dth[:, 0] += cnt(b[0], 1) + cnt(c[0], 2)
        dth[:, 1] += cnt(b[1], 1) + cnt(c[1], 2)
        dth[:, 2] += cnt(e[0], 3) + cnt(g[0], 4)
        dth[:, 3] += cnt(e[1], 3) + cnt(g[1], 4)
        B2, B1 = B1, cur
        F[t] = None
    pack = [torch.cat([M[p, :l1[p], W:W + l2[p]].reshape(-1) for p in range(n)]) for M in (OUT, POST)]
    return Z, pack[0], dth, pack[1]


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("scores", "softdp", "posterior"):
        return None         # hit lists: whole numbers, or the statistics of a whole search
    q, d = _pair_sets(case, seed)
    if kind == "scores":
        return _scores64(q, d)
    S, theta, w = _pair_inputs(case, seed, q, d)
    Z, dS, dth, post = _softdp64(q, d, S, theta)
    wd = w.double()
    size = torch.from_numpy((q.lengths().astype(np.int64) * d.lengths())).to(S.device)
    dS = dS * torch.repeat_interleave(wd, size)
    if kind == "softdp":
        return {"logZ": Z, "dS": dS, "dtheta": (dth * wd[:, None]).sum(0)}
    return {"logZ": Z, "dS": dS, "dtheta": dth * wd[:, None], "post": post}
