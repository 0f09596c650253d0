/*
 * c2_sdp.hip -- differentiable soft DP for gfx950: log-sum-exp forward and
 * its hand-written adjoint.  No reference counterpart.
 *
 * Model: the MAP forward model of the reference (ExecMAPDP_Fwd_Unroll32x,
 * cumapdp/CuBatchMAPDP_fwd.cu:291-372) with exact log-sum-exp: per cell the
 * states MM MI IM DN ND,
 *   MM = log(1 + e^{MI'+t+c+s} + e^{IM'+t+c+s} + e^{DN'+t+c+s} + e^{ND'+t+c+s} + e^{MM'+t+s})
 *   MI = lse(MM^ + t + o_I, MI^ + t + e_I)      IM = lse(MM< + t + o_I, IM< + t + e_I)
 *   DN = lse(MM^ + t + o_D, DN^ + t + e_D)      ND = lse(MM< + t + o_D, ND< + t + e_D)
 * (' diagonal, ^ up, < left; t the profile transitions; theta = (o_I, e_I,
 * o_D, e_D, c) five global log-offsets), row -1 = (MM 0, others -99), column
 * -1 = the MAP pass's boundary vectors, log Z = log sum_ij e^{MM(i,j)}.
 * Adjoint: the outside recursion B over the same terms in reverse;
 *   dlogZ/dS(i,j)   = e^{B_MM(i,j) - Z} (e^{F_MM(i,j)} - 1)
 *   dlogZ/dtheta_k  = sum of e^{F_src + term + B_dst - Z} over class-k terms
 *   posterior MM    = e^{F_MM + B_MM - Z}.
 * Arithmetic is base 2 inside (inputs scaled by log2 e once), with the
 * hardware exp2/log2.
 *
 * Decomposition: a pair is cut into stripes of 64 query rows, one wave per
 * stripe, lane l owning row l and processing column t-l at step t, the row
 * above arriving from lane l-1 by DPP wave_shr:1 (forward) and the row below
 * from lane l+1 by wave_shl:1 (adjoint).  A workgroup takes a band of up to 4
 * stripes that advance in lockstep, passing their boundary row through LDS.
 * Bands of one pair run in different workgroups at once: the boundary row goes through
 * memory as words that a launch first sets to a value no state has, so a
 * word is its own arrival flag and the band after polls 64 columns at a time
 * (agent-scope relaxed atomics, no fences).  Workgroups take (pair, band)
 * items from a counter in the order of the dependences, so the band a
 * workgroup waits for is always held by one that runs already.
 * The forward either stores all five states of every cell (K = 0) or only
 * the wave state every K steps (K divides 64); the adjoint then recomputes
 * each K-step segment from its checkpoint into per-wave scratch and sweeps
 * it backwards (sqrt(L) checkpointing).
 *
 * What bounds it: the sweep's chain of dependent steps, with too few waves to
 * hide it.  Per cell 16 (forward) and 21 (adjoint) transcendentals, of two
 * issue slots each, and about 115 and 155 other vector instructions; counted
 * on 1,024 pairs of 50-600, the vector units are busy 38% (forward) and 31%
 * (adjoint) of the time, with 2.6 and 1.8 waves per SIMD that spend 71% of
 * theirs waiting; on 24 pairs of 2,000-5,000 with checkpoints 19% and 17%,
 * with 0.8 waves.  No step loads what it uses: a profile's transitions pass
 * through LDS, scores, stored states and gradients go four columns at a time
 * a group ahead, and the terms that leave the matrix's edges are added after
 * the sweep.  One row per lane: the padding of a pair's last stripe is
 * at most 63 rows, and a step's chain is one cell.  Every cell's operations
 * and their order are those of the one-workgroup-per-pair sweep.  Measured
 * (before: stripes of 320 rows, one workgroup per pair, inputs loaded in the
 * step that used them): 1,024 pairs of 50-600, forward + adjoint 8.01 -> 3.86
 * ms; 24 pairs of 2,000-5,000 with checkpoints 143.7 -> 22.2 ms.
 */
#include <algorithm>
#include <type_traits>
#include "c2_dev.h"
#include "c2_kernels.h"

namespace {

constexpr float L2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;
constexpr float NEG = -1.0e30f;

__device__ __forceinline__ float ex2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float lg2(float x) { return __builtin_amdgcn_logf(x); }
__device__ __forceinline__ float lse2(float a, float b)
{
    return fmaxf(a, b) + lg2(1.0f + ex2(-fabsf(a - b)));
}

/* log-sum-exp of two terms as (max, e^{a-max}, e^{b-max}) with one exp2 */
__device__ __forceinline__ float lse_parts(float a, float b, float& fa, float& fb)
{
    const float e = ex2(-fabsf(a - b));
    const bool ab = a >= b;
    fa = ab ? 1.0f : e;
    fb = ab ? e : 1.0f;
    return fmaxf(a, b);
}

struct Th { float oi, ei, od, ed, cl; };

__device__ __forceinline__ S5 s5_fill(float mm, float rest)
{
    S5 s; s.mm = mm; s.mi = s.im = s.dn = s.nd = rest; return s;
}

/* transitions of query/profile row i in the MAP forward caching (MI, II at i+1), base 2 */
__device__ __forceinline__ void ld_trn(const float* T, int64_t ntr, int64_t base, int i, float t[7])
{
    t[0] = T[0 * ntr + base + i] * L2E;
    t[1] = T[1 * ntr + base + i + 1] * L2E;
    t[2] = T[2 * ntr + base + i] * L2E;
    t[3] = T[3 * ntr + base + i] * L2E;
    t[4] = T[4 * ntr + base + i + 1] * L2E;
    t[5] = T[5 * ntr + base + i] * L2E;
    t[6] = T[6 * ntr + base + i] * L2E;
}

/* Row-major S, dS and posterior blocks are read and written four columns at
 * a time: at anti-diagonal step t lane l holds column t-l of its row, so the
 * 4 steps of an aligned group (t = 4m..4m+3) cover 4 consecutive columns of
 * the row, one 16-byte access; the step loops are unrolled by four, so a
 * step's word is a fixed register.  Lanes at a row's two ends take single
 * words (clamped into the row when read). */
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef double f64u __attribute__((aligned(4)));

__device__ __forceinline__ f4u grp_load(const float* row, int c0, int L2)
{
    f4u v;
    if (c0 >= 0 && c0 + 3 < L2) {
        v = *(const f4u*)(row + c0);
    } else {
        v.x = row[min(max(c0, 0), L2 - 1)]; v.y = row[min(max(c0 + 1, 0), L2 - 1)];
        v.z = row[min(max(c0 + 2, 0), L2 - 1)]; v.w = row[min(max(c0 + 3, 0), L2 - 1)];
    }
    return v;
}
__device__ __forceinline__ void grp_store(float* row, int c0, int L2, const f4u& v)
{
    if (c0 >= 0 && c0 + 3 < L2) {
        *(f4u*)(row + c0) = v;
    } else {
        if (c0 >= 0 && c0 < L2) row[c0] = v.x;
        if (c0 + 1 >= 0 && c0 + 1 < L2) row[c0 + 1] = v.y;
        if (c0 + 2 >= 0 && c0 + 2 < L2) row[c0 + 2] = v.z;
        if (c0 + 3 >= 0 && c0 + 3 < L2) row[c0 + 3] = v.w;
    }
}

/* words handed from one workgroup to another: WAITING until written; a
 * state with those bits (a NaN some score carried in) goes as the plain NaN */
constexpr uint32_t WAITING = 0xFFFFFFFFu;
__device__ __forceinline__ void xput(float* p, float v)
{
    uint32_t u = __float_as_uint(v);
    if (u == WAITING) u = 0x7FC00000u;
    __hip_atomic_store((uint32_t*)p, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t xget(const float* p)
{
    return __hip_atomic_load((const uint32_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
/* N rows (ld apart) of one column per lane with want set, into LDS
 * dst[lane][n]; waits until every word has arrived.  The writer runs already
 * (see take_item) and waits for nothing of this workgroup's */
template <int N>
__device__ __forceinline__ void xwait(const float* p, int ld, bool want, float (*dst)[N], int lane)
{
    uint32_t v[N];
    for (;;) {
        bool ready = true;
#pragma unroll
        for (int n = 0; n < N; n++) v[n] = 0u;
        if (want) {
#pragma unroll
            for (int n = 0; n < N; n++) { v[n] = xget(p + (int64_t)n * ld); ready = ready && v[n] != WAITING; }
        }
        if (__ballot(!ready) == 0) break;
        __builtin_amdgcn_s_sleep(8);
    }
#pragma unroll
    for (int n = 0; n < N; n++) dst[lane][n] = __uint_as_float(v[n]);
    wave_lds_sync();
}

/* the workgroup's next item: from the launch's counter (items depend on
 * earlier ones), or a fixed stride (no pair has a second band) */
__device__ __forceinline__ int take_item(unsigned* head, int prev, int* slot)
{
    if (!head) return prev < 0 ? (int)blockIdx.x : prev + (int)gridDim.x;
    __syncthreads();
    if (threadIdx.x == 0) *slot = (int)atomicAdd(head, 1u);
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*slot);
}

__device__ __forceinline__ Th load_theta(const float* theta)
{
    Th t;
    t.oi = theta[0] * L2E; t.ei = theta[1] * L2E; t.od = theta[2] * L2E;
    t.ed = theta[3] * L2E; t.cl = theta[4] * L2E;
    return t;
}

/* row -1 of the matrix */
__device__ __forceinline__ S5 s5_top() { return s5_fill(0.0f, -99.0f * L2E); }

/* a wave's window of the profile's transitions (base 2): two blocks of 64
 * columns, column c at slot c & 127, 12 words apart (two 16-byte reads, the 8
 * lanes of a read on distinct banks).  A block is loaded into registers half
 * a block ahead of its first step, so that no step waits for memory (on this
 * chip a load's wait also waits for every older store) */
constexpr int TW = 12;
struct Col { f4 a, b; };
struct TrnWin {
    float* w;
    float v[7];
    __device__ __forceinline__ void fetch(const SdpArgs& a, int64_t db, int blk, int L2, int lane)
    {
        ld_trn(a.dtr, a.dntr, db, min(max(64 * blk + lane, 0), L2 - 1), v);
    }
    __device__ __forceinline__ void put(int blk, int lane)
    {
        f4* p = (f4*)(w + (((64 * blk) & 127) + lane) * TW);
        p[0] = f4{v[0], v[1], v[2], v[3]}; p[1] = f4{v[4], v[5], v[6], 0.0f};
        wave_lds_sync();
    }
    __device__ __forceinline__ Col get(int c) const
    {
        const f4* p = (const f4*)(w + (c & 127) * TW);
        Col r; r.a = p[0]; r.b = p[1];
        return r;
    }
};

/* wave state of the forward sweep of one stripe */
struct FwdState {
    S5 H;         /* the lane's row at its current column */
    S5 U;         /* the row above there, and its MM and MI + the row's MM transition, */
    float um, ui; /* which start the cell's MI terms now and its MM terms a step later */
};

/* a cell (the additions of each term in the model's order) */
__device__ __forceinline__ S5 fcell(const S5& dg, float dgm, float dgi, const FwdState& w, const float* q, const Col& d,
                                    float s, const Th& th)
{
    const float d0 = d.a[0], d1 = d.a[1], d2 = d.a[2], d3 = d.a[3], d4 = d.b[0], d5 = d.b[1], d6 = d.b[2];
    const float a0 = dgi + d3 + th.cl + s;
    const float a1 = dg.im + q[3] + d0 + th.cl + s;
    const float a2 = dg.dn + q[5] + d0 + th.cl + s;
    const float a3 = dg.nd + q[0] + d5 + th.cl + s;
    const float a4 = dgm + d0 + s;
    const float m = fmaxf(fmaxf(fmaxf(a0, a1), fmaxf(a2, a3)), fmaxf(a4, 0.0f));
    const float sum = ex2(a0 - m) + ex2(a1 - m) + ex2(a2 - m) + ex2(a3 - m) + ex2(a4 - m) + ex2(-m);
    S5 n;
    n.mm = m + lg2(sum);
    n.mi = lse2(w.um + d1 + th.oi, w.ui + d4 + th.ei);
    n.im = lse2(w.H.mm + q[1] + d0 + th.oi, w.H.im + q[4] + d0 + th.ei);
    n.dn = lse2(w.U.mm + q[2] + th.od, w.U.dn + q[6] + th.ed);
    n.nd = lse2(w.H.mm + d2 + th.od, w.H.nd + d6 + th.ed);
    return n;
}

__device__ __forceinline__ S5 ld_col(const float* v)
{
    S5 s; s.mm = v[0] * L2E; s.mi = v[1] * L2E; s.im = v[2] * L2E; s.dn = v[3] * L2E; s.nd = v[4] * L2E;
    return s;
}

/* before the first step: a lane's state is the column left of the matrix
 * until it enters its first column, which is what the row below sees as its
 * diagonal there (rows r % 32 == 31 excepted: theirs is row -1's); lane 0
 * starts under row -1 */
__device__ __forceinline__ void fwd_init(const SdpArgs& a, const SdpPair& P, int r, FwdState& w)
{
    w.H = ld_col(a.qll + ((int64_t)a.qdist[P.q] + min(r, P.L1 - 1)) * 5);
    w.U = s5_top();
}

/* one step of the lane: the row above arrives (lane l takes lane l-1's row,
 * lane 0 the stripe's top boundary tp), the one it had becomes the diagonal;
 * ALL: every lane is inside the matrix past column 0 */
template <bool ALL>
__device__ __forceinline__ void fwd_step(const float* q, bool m31, FwdState& w, int c, int L2, const Col& d, float sc,
                                         const S5& tp, const Th& th)
{
    S5 dg = w.U;
    float dgm = w.um, dgi = w.ui;
    w.U.mm = wave_shr1(w.H.mm, tp.mm);
    w.U.mi = wave_shr1(w.H.mi, tp.mi);
    w.U.im = wave_shr1(w.H.im, tp.im);
    w.U.dn = wave_shr1(w.H.dn, tp.dn);
    w.U.nd = wave_shr1(w.H.nd, tp.nd);
    w.um = w.U.mm + q[0];
    w.ui = w.U.mi + q[0];
    if (ALL) {
        w.H = fcell(dg, dgm, dgi, w, q, d, sc * L2E, th);
    } else if (c >= 0 && c < L2) {
        if (c == 0 && m31) { dg = s5_top(); dgm = dg.mm + q[0]; dgi = dg.mi + q[0]; }
        w.H = fcell(dg, dgm, dgi, w, q, d, sc * L2E, th);
    }
}
__device__ __forceinline__ S5 s5_at(const float* o, int ld)
{
    S5 s; s.mm = o[0]; s.mi = o[ld]; s.im = o[2 * ld]; s.dn = o[3 * ld]; s.nd = o[4 * ld];
    return s;
}

/* the last row of stripe s as the stripe below reads it ([5][L2]): between
 * bands in the hand-off region, inside a band (kept for the adjoint's
 * recomputation) in the pair's own */
__device__ __forceinline__ float* last_row(const SdpArgs& a, const SdpPair& P, int s, int NW)
{
    return (s + 1) % NW == 0 ? a.ws + P.boff + (int64_t)((s + 1) / NW - 1) * 5 * P.L2
                             : a.ws + P.hoff + (int64_t)s * 5 * P.L2;
}

/* four steps' states of the lane: a group's block is [5][64 lanes][4].  The
 * workspace is the caller's, at any float's address: its words are accessed
 * as such (the device takes 16-byte accesses at 4-byte addresses, and no
 * instruction differs for an aligned workspace) */
struct Quad { f4 mm, mi, im, dn, nd; };
__device__ __forceinline__ void quad_set(Quad& q, int u, const S5& s)
{
    q.mm[u] = s.mm; q.mi[u] = s.mi; q.im[u] = s.im; q.dn[u] = s.dn; q.nd[u] = s.nd;
}
__device__ __forceinline__ S5 quad_get(const Quad& q, int u)
{
    S5 s; s.mm = q.mm[u]; s.mi = q.mi[u]; s.im = q.im[u]; s.dn = q.dn[u]; s.nd = q.nd[u];
    return s;
}
__device__ __forceinline__ void quad_put(float* blk, int lane, const Quad& q)
{
    f4u* p = (f4u*)blk + lane;
    p[0] = q.mm; p[64] = q.mi; p[128] = q.im; p[192] = q.dn; p[256] = q.nd;
}
__device__ __forceinline__ void quad_load(const float* blk, int lane, Quad& q)
{
    const f4u* p = (const f4u*)blk + lane;
    q.mm = p[0]; q.mi = p[64]; q.im = p[128]; q.dn = p[192]; q.nd = p[256];
}
constexpr int QUAD = 5 * 64 * 4;      /* floats of a group's block */

/* checkpoint of the wave state: H, U (5 floats each) */
constexpr int CKPT = 10 * 64;
__device__ __forceinline__ void put_ckpt(float* base, int lane, const FwdState& w)
{
    const S5* v[2] = {&w.H, &w.U};
#pragma unroll
    for (int i = 0; i < 2; i++) {
        float* b = base + i * 320 + lane;
        b[0] = v[i]->mm; b[64] = v[i]->mi; b[128] = v[i]->im; b[192] = v[i]->dn; b[256] = v[i]->nd;
    }
}
__device__ __forceinline__ void get_ckpt(const float* base, int lane, FwdState& w)
{
    w.H = s5_at(base + lane, 64); w.U = s5_at(base + 320 + lane, 64);
}

/* sums t 2^m of the matrix's e^MM, joined */
__device__ __forceinline__ void zsum(float& m, float& t, float om, float os)
{
    const float mm = fmaxf(m, om);
    t = t * ex2(m - mm) + os * ex2(om - mm);
    m = mm;
}

/* forward of one (pair, band) item after another; the waves of a band are
 * 68 steps apart, so that the columns t0..t0+3 a wave's group needs of the
 * row above were written a group ago: one barrier per group.  Rows cross in
 * LDS rings of 16 columns */
constexpr int LAG = 68;
__global__ __launch_bounds__(64 * C2_SDP_BAND) void k_sdp_fwd(SdpArgs a)
{
    __shared__ __align__(16) float hx[C2_SDP_BAND][16][5];
    __shared__ __align__(16) float win[C2_SDP_BAND][128 * TW];
    __shared__ __align__(16) float tb[64][5];          /* the row above the band, 64 columns */
    __shared__ float wz[C2_SDP_BAND][2];
    __shared__ int tick;
    const int lane = threadIdx.x & 63, NW = blockDim.x >> 6;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const Th th = load_theta(a.theta);
    for (int it = take_item(a.head, -1, &tick); it < a.nitems; it = take_item(a.head, it, &tick)) {
        const int pi = __builtin_amdgcn_readfirstlane(a.items[it].x), b = __builtin_amdgcn_readfirstlane(a.items[it].y);
        const SdpPair P = a.pairs[pi];
        const int ns = P.ns, L2 = P.L2, nsteps = L2 + 63;
        const int64_t db = (int64_t)a.ddist[P.p] + P.p;
        const int nwb = min(NW, ns - b * NW);
        const bool have = wv < nwb;
        const int s = b * NW + min(wv, nwb - 1);
        const bool out = wv == nwb - 1 && s + 1 < ns;    /* its last row leaves the workgroup */
        const int r = s * 64 + lane, rc = min(r, P.L1 - 1);
        const bool valid = r < P.L1, m31 = (r & 31) == 31;
        const float* S = a.S + P.soff + (int64_t)rc * L2;
        float* store = a.ws + P.foff;
        float q[7];
        ld_trn(a.qtr, a.qntr, (int64_t)a.qdist[P.q] + P.q, rc, q);
        FwdState w;
        fwd_init(a, P, r, w);
        w.um = w.U.mm + q[0]; w.ui = w.U.mi + q[0];
        /* sum of 2^(F_MM - zr), the reference raised when a term would leave it by
         * 2^64, and the largest F_MM */
        float zr = 0.0f, zs = 0.0f, zm = NEG;
        f4u sc = grp_load(S, -lane, L2), sn = sc;
        TrnWin tw;
        tw.w = win[wv];
        tw.fetch(a, db, 0, L2, lane);
        tw.put(0, lane);
        const int TT = nsteps + LAG * (nwb - 1);
        for (int T0 = 0; T0 < TT; T0 += 4) {
            const int t0 = T0 - LAG * wv;               /* this wave's group */
            if (have && t0 >= 0 && t0 < nsteps) {
                sc = sn;
                if (t0 + 4 < nsteps) sn = grp_load(S, t0 + 4 - lane, L2);
                if ((t0 & 15) == 0) {
                    if (a.K > 0 && t0 > 0 && (t0 & (a.K - 1)) == 0)
                        put_ckpt(store + ((int64_t)s * P.ncp + t0 / a.K) * CKPT, lane, w);
                    if ((t0 & 63) == 32) tw.fetch(a, db, (t0 >> 6) + 1, L2, lane);
                    if ((t0 & 63) == 0) {
                        if (t0 > 0) tw.put(t0 >> 6, lane);
                        if (wv == 0 && b > 0 && t0 < L2)
                            xwait<5>(last_row(a, P, s - 1, NW) + t0 + lane, L2, t0 + lane < L2, tb, lane);
                    }
                }
                /* the row above at columns t0 .. t0+3 */
                float tp[20];
                if (s == 0) {
                    const S5 z = s5_top();
#pragma unroll
                    for (int i = 0; i < 20; i++) tp[i] = (i % 5) ? z.mi : z.mm;
                } else {
                    const f4* o = (const f4*)(wv > 0 ? &hx[wv - 1][t0 & 15][0] : &tb[t0 & 63][0]);
#pragma unroll
                    for (int i = 0; i < 5; i++) {
                        const f4 x = o[i];
#pragma unroll
                        for (int j = 0; j < 4; j++) tp[4 * i + j] = x[j];
                    }
                }
                Quad qd;
                auto step = [&](auto ALLC, auto UC) __attribute__((always_inline)) {
                    constexpr bool ALL = decltype(ALLC)::value;
                    constexpr int u = decltype(UC)::value;
                    const int c = t0 + u - lane;
                    const S5 top = s5_at(tp + 5 * u, 1);
                    fwd_step<ALL>(q, m31, w, c, L2, tw.get(c), sc[u], top, th);
                    const float f = valid && (ALL || (c >= 0 && c < L2)) ? w.H.mm : NEG;
                    float e = f - zr;
                    zm = fmaxf(zm, f);
                    if (e > 64.0f) { zs *= ex2(-e); zr = f; e = 0.0f; }
                    zs += ex2(e);
                    quad_set(qd, u, w.H);
                };
                using std::integral_constant;
                if (t0 >= 64 && t0 + 3 < L2) {
                    step(std::true_type{}, integral_constant<int, 0>{}); step(std::true_type{}, integral_constant<int, 1>{});
                    step(std::true_type{}, integral_constant<int, 2>{}); step(std::true_type{}, integral_constant<int, 3>{});
                } else {
                    step(std::false_type{}, integral_constant<int, 0>{}); step(std::false_type{}, integral_constant<int, 1>{});
                    step(std::false_type{}, integral_constant<int, 2>{}); step(std::false_type{}, integral_constant<int, 3>{});
                }
                if (a.K == 0) quad_put(store + ((int64_t)s * ((nsteps + 3) >> 2) + (t0 >> 2)) * QUAD, lane, qd);
                if (lane == 63 && s + 1 < ns) {
                    /* the row's columns t0-63 .. t0-60 */
                    float* h = nullptr;
                    if (out || a.K > 0) h = last_row(a, P, s, NW);
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const int c = t0 + u - 63;
                        if (c < 0 || c >= L2) continue;
                        const S5 e = quad_get(qd, u);
                        if (out) {
                            xput(h + c, e.mm); xput(h + (int64_t)L2 + c, e.mi); xput(h + (int64_t)2 * L2 + c, e.im);
                            xput(h + (int64_t)3 * L2 + c, e.dn); xput(h + (int64_t)4 * L2 + c, e.nd);
                        } else {
                            float* o = hx[wv][c & 15];
                            o[0] = e.mm; o[1] = e.mi; o[2] = e.im; o[3] = e.dn; o[4] = e.nd;
                            if (a.K > 0) {
                                h[c] = e.mm; h[(int64_t)L2 + c] = e.mi; h[(int64_t)2 * L2 + c] = e.im;
                                h[(int64_t)3 * L2 + c] = e.dn; h[(int64_t)4 * L2 + c] = e.nd;
                            }
                        }
                    }
                }
            }
            __syncthreads();
        }
        /* the item's sum: deterministic xor-butterfly of the lanes' (maximum,
         * scaled sum), then the waves in order */
        zs = zm == NEG ? zs : zs * ex2(zr - zm);      /* (no cell of the lane's: zs is 0) */
        for (int off = 32; off >= 1; off >>= 1) {
            const float om = __shfl_xor(zm, off), os = __shfl_xor(zs, off);
            const float m = fmaxf(zm, om);
            zs = zs * ex2(zm - m) + os * ex2(om - m);
            zm = m;
        }
        if (lane == 0) { wz[wv][0] = zm; wz[wv][1] = zs; }
        __syncthreads();
        if (threadIdx.x == 0) {
            float m = wz[0][0], t = wz[0][1];
            for (int k = 1; k < nwb; k++) zsum(m, t, wz[k][0], wz[k][1]);
            if (a.head) {
                float* z = a.ws + a.zpart_off + 2 * (int64_t)(P.i0 + b);
                z[0] = m; z[1] = t;
            } else {
                a.logZ[pi] = (m + lg2(t)) * LN2;
            }
        }
        __syncthreads();
    }
}

/* adjoint: the forward's stripes and bands, bottom-up; inside a band wave w
 * runs behind wave w+1 in the reverse sweep, which hands its row (B_MM+S,
 * B_MI, B_DN) up through a double-buffered LDS slot.  With every cell stored
 * the waves are 68 steps apart with one barrier per group, as in the
 * forward.  With checkpoints (CK) the sweep goes in phases of K steps (a
 * divisor of 64): every wave recomputes its phase's forward states from the
 * checkpoint into its own scratch, then the band takes K reverse steps, 64
 * steps apart (so the waves recompute at the same time) with a barrier per
 * step. */
template <bool CK>
__global__ __launch_bounds__(64 * C2_SDP_BAND) void k_sdp_adj(SdpArgs a)
{
    __shared__ float hb[2][C2_SDP_BAND][4][3];
    __shared__ __align__(16) float win[C2_SDP_BAND][128 * TW];
    __shared__ float bb[64][3];                      /* the row below the band, one phase's columns */
    __shared__ __align__(16) float tq[CK ? C2_SDP_BAND : 1][64][5];          /* the recomputation's row above, per wave */
    __shared__ double wacc[C2_SDP_BAND][5];
    __shared__ int tick;
    const int lane = threadIdx.x & 63, NW = blockDim.x >> 6;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const Th th = load_theta(a.theta);
    const int KK = CK ? a.K : 64;
    constexpr int lagw = CK ? 64 : LAG;
    float* scr = a.ws + a.scr_off + (int64_t)(blockIdx.x * NW + wv) * (a.K >> 2) * QUAD;
    for (int it = take_item(a.head, -1, &tick); it < a.nitems; it = take_item(a.head, it, &tick)) {
        const int pi = __builtin_amdgcn_readfirstlane(a.items[it].x), b = __builtin_amdgcn_readfirstlane(a.items[it].y);
        const SdpPair P = a.pairs[pi];
        const int ns = P.ns, L2 = P.L2, nsteps = L2 + 63, ngrp = (nsteps + 3) >> 2;
        const float Z = a.logZ[pi] * L2E;
        const float g = a.gZ ? a.gZ[pi] : 1.0f;
        const int64_t db = (int64_t)a.ddist[P.p] + P.p;
        const int64_t qb = (int64_t)a.qdist[P.q] + P.q;
        const int nwb = min(NW, ns - b * NW);
        const bool have = wv < nwb;
        const int s = b * NW + min(wv, nwb - 1);
        const bool below = s + 1 < ns;                   /* a stripe follows */
        const bool far = below && wv == nwb - 1;         /* in another workgroup */
        float* frow = a.ws + P.aoff + (int64_t)b * 3 * L2;   /* this band's first row [3][L2] */
        const int r = s * 64 + lane, rc = min(r, P.L1 - 1);
        const bool valid = r < P.L1, m31 = (r & 31) == 31;
        const int64_t ro = P.soff + (int64_t)rc * L2;
        const float* S = a.S + ro;
        const float* store = a.ws + P.foff;
        float qs[7], qr[7];                      /* transitions of the lane's row and the one below */
        ld_trn(a.qtr, a.qntr, qb, rc, qs);
        ld_trn(a.qtr, a.qntr, qb, min(r + 1, P.L1 - 1), qr);
        S5 cur = s5_fill(NEG, NEG);              /* B at (r, c+1); mm carries + S */
        /* B_MM+S, B_MI, B_DN of the row below at the next column (sh), B_MM+S a
         * column further (shpbs) */
        float shbs = NEG, shmi = NEG, shdn = NEG, shpbs = NEG;
        Col dx;                                  /* transitions of column c+1 */
        dx.a = dx.b = f4{0.0f, 0.0f, 0.0f, 0.0f};
        /* column 0's B_MM+S, B_IM, B_ND: the edge terms after the sweep */
        float e0bs = NEG, e0im = NEG, e0nd = NEG;
        double acc0 = 0.0, acc1 = 0.0, acc2 = 0.0, acc3 = 0.0, acc4 = 0.0;
        const int tl = nsteps - 1;
        f4u sc = grp_load(S, (tl & ~3) - lane, L2), sn = sc;
        Quad F, Fn;
        if (!CK) quad_load(store + ((int64_t)s * ngrp + (tl >> 2)) * QUAD, lane, Fn);
        TrnWin tw;
        tw.w = win[wv];
        tw.fetch(a, db, tl >> 6, L2, lane);
        tw.put(tl >> 6, lane);
        tw.fetch(a, db, (tl >> 6) - 1, L2, lane);
        tw.put((tl >> 6) - 1, lane);
        /* groups of the wave, last first, in phases of KK steps over 0..nsteps */
        const int nsegp = nsteps / KK + 1;
        const int tend = nsegp * KK;                     /* one past the first step taken */
        const int TT = tend + lagw * (nwb - 1);
        float f0 = 0.0f, f1 = 0.0f, f2 = 0.0f, f3 = 0.0f, f4_ = 0.0f;
        for (int T0 = 0; T0 < TT; T0 += 4) {
            const int g0 = tend - 4 - T0 + lagw * (nwb - 1 - wv);      /* the group's first column step */
            const int par = (T0 >> 2) & 1;
            const bool on = have && g0 >= 0 && g0 < tend;
            if (on) {
                if ((g0 & 63) == 28 && g0 < nsteps) tw.fetch(a, db, (g0 >> 6) - 2, L2, lane);
                if ((g0 & 63) == 60 && g0 + 4 < nsteps) {
                    /* block g0/64 + 1 is done with; the one before this group's goes in */
                    if (g0 + 36 >= nsteps) tw.fetch(a, db, (g0 >> 6) - 1, L2, lane);
                    tw.put((g0 >> 6) - 1, lane);
                }
                if ((g0 & (KK - 1)) == KK - 4) {
                    /* a phase starts: [p0, p0 + KK) */
                    const int p0 = g0 & ~(KK - 1);
                    if (CK && p0 < nsteps) {
                        /* its forward states, recomputed from the checkpoint */
                        const int t1 = min(nsteps, p0 + KK);
                        FwdState w;
                        const float* top = s > 0 ? last_row(a, P, s - 1, NW) : nullptr;
                        if (s > 0) {
                            const int c = min(p0 + lane, L2 - 1);
#pragma unroll
                            for (int n = 0; n < 5; n++) tq[wv][lane][n] = top[(int64_t)n * L2 + c];
                        } else {
                            const S5 z = s5_top();
                            tq[wv][lane][0] = z.mm;
#pragma unroll
                            for (int n = 1; n < 5; n++) tq[wv][lane][n] = z.mi;
                        }
                        if (p0 == 0) {
                            fwd_init(a, P, r, w);
                        } else {
                            get_ckpt(store + ((int64_t)s * P.ncp + p0 / KK) * CKPT, lane, w);
                        }
                        w.um = w.U.mm + qs[0]; w.ui = w.U.mi + qs[0];
                        /* the window holds the phase's columns (its block and the one before) */
                        wave_lds_sync();
                        f4u rs, rn = grp_load(S, p0 - lane, L2);
                        for (int tg = p0; tg < t1; tg += 4) {
                            rs = rn;
                            rn = grp_load(S, tg + 4 - lane, L2);
                            Quad q;
                            const bool all = tg >= 64 && tg + 3 < L2;
#pragma unroll
                            for (int u = 0; u < 4; u++) {
                                const int c = tg + u - lane;
                                const S5 tp = s5_at(&tq[wv][tg + u - p0][0], 1);
                                if (all) fwd_step<true>(qs, m31, w, c, L2, tw.get(c), rs[u], tp, th);
                                else fwd_step<false>(qs, m31, w, c, L2, tw.get(c), rs[u], tp, th);
                                quad_set(q, u, w.H);
                            }
                            quad_put(scr + (int64_t)((tg - p0) >> 2) * QUAD, lane, q);
                        }
                        __threadfence_block();
                        quad_load(scr + (int64_t)((t1 - 1 - p0) >> 2) * QUAD, lane, Fn);
                    }
                    if (far) {
                        /* this phase takes the row below at columns p0-64 .. p0+KK-65 */
                        const int c = p0 - 64 + lane;
                        xwait<3>(frow + (int64_t)3 * L2 + c, L2, lane < KK && c >= 0 && c < L2, bb, lane);
                    }
                    /* the phase before's parameter-gradient sums, FP32 over at most
                     * KK terms per lane, join the item's in FP64 */
                    acc0 += (double)f0; acc1 += (double)f1; acc2 += (double)f2; acc3 += (double)f3; acc4 += (double)f4_;
                    f0 = f1 = f2 = f3 = f4_ = 0.0f;
                }
                if (g0 < nsteps) {
                    sc = sn; F = Fn;
                    if (g0 >= 4) {
                        sn = grp_load(S, g0 - 4 - lane, L2);
                        if (!CK) quad_load(store + ((int64_t)s * ngrp + ((g0 - 4) >> 2)) * QUAD, lane, Fn);
                        else if (g0 & (KK - 1)) quad_load(scr + (int64_t)(((g0 - 4) & (KK - 1)) >> 2) * QUAD, lane, Fn);
                    }
                }
            }
            f4u dv, pv;
            f4 ub, ui, ud;                       /* lane 0's B_MM+S, B_MI, B_DN */
#pragma unroll
            for (int u = 3; u >= 0; u--) {
                const int t = g0 + u;
                if (on && t < nsteps) {
                    const int c = t - lane;
                    const Col dc = tw.get(c);
                    if (c >= 0 && c < L2 && valid) {
                        const S5 rt = cur;                              /* (r, c+1) */
                        const float dgbs = shpbs;                       /* (r+1, c+1) */
                        const float x0 = dx.a[0], gq = dgbs + qr[0], mq = shmi + qr[0];
                        /* MM: end, MM->MM, MM->MI, MM->IM, MM->DN, MM->ND */
                        const float m1 = gq + x0;
                        const float m2 = mq + dc.a[1] + th.oi;
                        const float m3 = rt.im + qs[1] + x0 + th.oi;
                        const float m4 = shdn + qr[2] + th.od;
                        const float m5 = rt.nd + dx.a[2] + th.od;
                        const float mm = fmaxf(fmaxf(fmaxf(m1, m2), fmaxf(m3, m4)), fmaxf(m5, 0.0f));
                        const float e2 = ex2(m2 - mm), e3 = ex2(m3 - mm), e4 = ex2(m4 - mm), e5 = ex2(m5 - mm);
                        const float sum6 = ex2(-mm) + ex2(m1 - mm) + e2 + e3 + e4 + e5;
                        const float bmm = mm + lg2(sum6);
                        /* gap states: two terms each, the larger one is e^0 = 1 */
                        float fi1, fi2, fj1, fj2, fd1, fd2, fn1, fn2;
                        /* MI: close, extend */
                        const float mi = lse_parts(gq + dx.a[3] + th.cl, mq + dc.b[0] + th.ei, fi1, fi2);
                        /* IM */
                        const float mj = lse_parts(dgbs + qr[3] + x0 + th.cl, rt.im + qs[4] + x0 + th.ei, fj1, fj2);
                        /* DN */
                        const float md = lse_parts(dgbs + qr[5] + x0 + th.cl, shdn + qr[6] + th.ed, fd1, fd2);
                        /* ND */
                        const float mn = lse_parts(gq + dx.b[1] + th.cl, rt.nd + dx.b[2] + th.ed, fn1, fn2);
                        const S5 f = quad_get(F, u);
                        const float wz = ex2(bmm - Z);
                        /* e^{F_MM + B_MM - Z} = e^{F_MM + mm - Z} * sum6 */
                        const float wm = ex2(f.mm + mm - Z), wi = ex2(f.mi + mi - Z), wj = ex2(f.im + mj - Z);
                        const float wd = ex2(f.dn + md - Z), wn = ex2(f.nd + mn - Z);
                        const float pmm = wm * sum6;
                        dv[u] = (pmm - wz) * g;
                        pv[u] = pmm;
                        f0 = fmaf(wm, e2 + e3, f0);
                        f2 = fmaf(wm, e4 + e5, f2);
                        f1 = fmaf(wi, fi2, fmaf(wj, fj2, f1));
                        f3 = fmaf(wd, fd2, fmaf(wn, fn2, f3));
                        f4_ = fmaf(wi, fi1, fmaf(wj, fj1, fmaf(wd, fd1, fmaf(wn, fn1, f4_))));
                        cur.mm = bmm + sc[u] * L2E;
                        cur.mi = mi + lg2(fi1 + fi2);
                        cur.im = mj + lg2(fj1 + fj2);
                        cur.dn = md + lg2(fd1 + fd2);
                        cur.nd = mn + lg2(fn1 + fn2);
                        if (c == 0) { e0bs = cur.mm; e0im = cur.im; e0nd = cur.nd; }
                    } else {
                        cur = s5_fill(NEG, NEG);
                    }
                    ub[u] = cur.mm; ui[u] = cur.mi; ud[u] = cur.dn;
                    if (CK && lane == 0 && wv > 0) {
                        float* o = hb[u & 1][wv][0];
                        o[0] = cur.mm; o[1] = cur.mi; o[2] = cur.dn;
                    }
                    dx = dc;
                }
                if (CK) __syncthreads();
                if (on && t >= 1 && t <= nsteps) {
                    /* the row below for step t-1: lane l+1's row, or for lane 63 the
                     * stripe below at column t-1-63 */
                    float obs = NEG, omi = NEG, odn = NEG;
                    const int cb = t - 1 - 63;
                    if (below && cb >= 0 && cb < L2) {
                        if (!far) {
                            const float* o = CK ? hb[u & 1][wv + 1][0] : hb[par ^ 1][wv + 1][u];
                            obs = o[0]; omi = o[1]; odn = o[2];
                        } else {
                            const int i = t & (KK - 1);
                            obs = bb[i][0]; omi = bb[i][1]; odn = bb[i][2];
                        }
                    }
                    shpbs = shbs;
                    shbs = wave_shl1(cur.mm, obs);
                    shmi = wave_shl1(cur.mi, omi);
                    shdn = wave_shl1(cur.dn, odn);
                }
            }
            if (on && g0 < nsteps) {
                /* the group's four columns go out */
                if (valid) {
                    grp_store(a.dS + ro, g0 - lane, L2, dv);
                    if (a.post) grp_store(a.post + ro, g0 - lane, L2, pv);
                }
                if (lane == 0) {
                    /* lane 0's row at columns g0 .. g0+3 */
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const int c = g0 + u;
                        if (c >= L2) continue;
                        const float xb = ub[u], xi = ui[u], xd = ud[u];
                        if (wv > 0) {
                            if (!CK) { float* o = hb[par][wv][u]; o[0] = xb; o[1] = xi; o[2] = xd; }
                        } else if (b > 0) {
                            xput(frow + c, xb); xput(frow + (int64_t)L2 + c, xi); xput(frow + (int64_t)2 * L2 + c, xd);
                        } else {
                            frow[c] = xb; frow[(int64_t)L2 + c] = xi; frow[(int64_t)2 * L2 + c] = xd;
                        }
                    }
                }
            }
            if (!CK) __syncthreads();
        }
        acc0 += (double)f0; acc1 += (double)f1; acc2 += (double)f2; acc3 += (double)f3; acc4 += (double)f4_;
        /* transitions whose source is the column left of the matrix or row -1,
         * counted at their destination */
        const float lp0 = -99.0f * L2E;
        if (have && valid) {
            float d0[7];
            ld_trn(a.dtr, a.dntr, db, 0, d0);
            const int64_t bi = ((int64_t)a.qdist[P.q] + r) * 5;
            const S5 lf = ld_col(a.qll + bi), dg = ld_col(a.qld + bi);
            acc0 += (double)ex2(lf.mm + qs[1] + d0[0] + th.oi + e0im - Z);
            acc1 += (double)ex2(lf.im + qs[4] + d0[0] + th.ei + e0im - Z);
            acc2 += (double)ex2(lf.mm + d0[2] + th.od + e0nd - Z);
            acc3 += (double)ex2(lf.nd + d0[6] + th.ed + e0nd - Z);
            acc4 += (double)(ex2(dg.mi + qs[0] + d0[3] + th.cl + e0bs - Z) + ex2(dg.im + qs[3] + d0[0] + th.cl + e0bs - Z) +
                             ex2(dg.dn + qs[5] + d0[0] + th.cl + e0bs - Z) + ex2(dg.nd + qs[0] + d0[5] + th.cl + e0bs - Z));
        }
        if (b == 0 && wv == 0) {
            /* row 0, its columns over the lanes (lane 0 of this wave wrote them) */
            __threadfence_block();
            float q0[7];
            ld_trn(a.qtr, a.qntr, qb, 0, q0);
            for (int c = lane; c < L2; c += 64) {
                float d[7];
                ld_trn(a.dtr, a.dntr, db, c, d);
                const float bs = frow[c], bmi = frow[(int64_t)L2 + c], bdn = frow[(int64_t)2 * L2 + c];
                acc0 += (double)ex2(q0[0] + d[1] + th.oi + bmi - Z);
                acc1 += (double)ex2(lp0 + q0[0] + d[4] + th.ei + bmi - Z);
                acc2 += (double)ex2(q0[2] + th.od + bdn - Z);
                acc3 += (double)ex2(lp0 + q0[6] + th.ed + bdn - Z);
                if (c > 0)
                    acc4 += (double)(ex2(lp0 + q0[0] + d[3] + th.cl + bs - Z) + ex2(lp0 + q0[3] + d[0] + th.cl + bs - Z) +
                                     ex2(lp0 + q0[5] + d[0] + th.cl + bs - Z) + ex2(lp0 + q0[0] + d[5] + th.cl + bs - Z));
            }
        }
        /* dtheta: fixed-order xor-butterfly in double, then the waves in order */
        for (int off = 32; off >= 1; off >>= 1) {
            acc0 += __shfl_xor(acc0, off); acc1 += __shfl_xor(acc1, off); acc2 += __shfl_xor(acc2, off);
            acc3 += __shfl_xor(acc3, off); acc4 += __shfl_xor(acc4, off);
        }
        if (lane == 0) {
            wacc[wv][0] = acc0; wacc[wv][1] = acc1; wacc[wv][2] = acc2; wacc[wv][3] = acc3; wacc[wv][4] = acc4;
        }
        __syncthreads();
        if (threadIdx.x < 5) {
            double t = 0.0;
            for (int k = 0; k < nwb; k++) t += wacc[k][threadIdx.x];
            if (a.head) ((f64u*)(a.ws + a.dpart_off))[(int64_t)5 * (P.i0 + b) + threadIdx.x] = t;
            else a.dth[(size_t)pi * 5 + threadIdx.x] = (float)(t * g);
        }
        __syncthreads();
    }
}

/* before a launch whose pairs have several bands: the item counter and the
 * hand-off rows */
__global__ __launch_bounds__(256) void k_sdp_begin(uint32_t* head, uint32_t* rows, int64_t n)
{
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i0 == 0) *head = 0u;
    for (int64_t i = i0; i < n; i += (int64_t)gridDim.x * blockDim.x) rows[i] = WAITING;
}
/* after it: the pairs' sums over their bands, in band order */
__global__ __launch_bounds__(256) void k_sdp_sums(SdpArgs a, int adjoint)
{
    const int pi = blockIdx.x * blockDim.x + threadIdx.x;
    if (pi >= a.npairs) return;
    const SdpPair P = a.pairs[pi];
    if (adjoint) {
        const f64u* d = (const f64u*)(a.ws + a.dpart_off) + (int64_t)5 * P.i0;
        const float g = a.gZ ? a.gZ[pi] : 1.0f;
        for (int j = 0; j < 5; j++) {
            double t = 0.0;
            for (int b = 0; b < P.nb; b++) t += d[5 * b + j];
            a.dth[(size_t)pi * 5 + j] = (float)(t * g);
        }
    } else {
        const float* z = a.ws + a.zpart_off + 2 * (int64_t)P.i0;
        float m = z[0], t = z[1];
        for (int b = 1; b < P.nb; b++) zsum(m, t, z[2 * b], z[2 * b + 1]);
        a.logZ[pi] = (m + lg2(t)) * LN2;
    }
}

/* score matrices of the prepared pairs from the raw profile fields:
 * S = log(sum_a q_a d_a / (0.5 (bq_a + bd_a))) - shift
 *     + ssswgt (sum_j p'_j QT[10j+int(9.999 p'_j)] + (p_H+0.1)(p'_H+0.1) 0.1111111 - 0.05),
 * QT(row)[g] = sum_i p_i T[10i+int(9.999 p_i)][g]
 * (CalcSM_Init_SMEMUnroll2x + CalcSM_SSSS_SMEMUnroll2x), the operations of
 * the search kernels.
 *
 * One workgroup per item of (pair, SC_ROWS query rows): the rows'
 * frequencies and SS tables go to LDS, and the waves take units of 16 rows x
 * 64 columns, a column's 20 weighted frequencies in a lane's registers, four
 * rows at a time (16-byte LDS reads); a row's 64 scores are one 256-byte
 * store.  Bound by VALU issue (about 55 operations a cell).  1,024 pairs of
 * 50-600 (108 M cells): 1.19 -> 0.25 ms (430 GCUPS); one workgroup per
 * pair re-read both profiles' 23 fields from memory for every cell.  Rows in
 * scalar registers (four or two at a time) spilled them and ran 0.36-0.40. */
constexpr int SC_ROWS = 32;

__global__ __launch_bounds__(256) void k_sdp_scores(SdpScoreArgs a)
{
    __shared__ __align__(16) float qt[30][SC_ROWS], qf[20][SC_ROWS];
    __shared__ __align__(16) float qh[SC_ROWS];
    __shared__ float w[20];
    const int pi = __builtin_amdgcn_readfirstlane(a.items[blockIdx.x].x);
    const int r0 = __builtin_amdgcn_readfirstlane(a.items[blockIdx.x].y);
    const SdpPair P = a.pairs[pi];
    const int nr = min(SC_ROWS, P.L1 - r0);
    const int64_t q0 = (int64_t)a.qdist[P.q] + r0, d0 = a.ddist[P.p];
    const bool ss_on = a.ssswgt > 0.0f;
    if (ss_on) {
        for (int i = threadIdx.x; i < 30 * SC_ROWS; i += blockDim.x) {
            const int g = i / SC_ROWS, r = i % SC_ROWS;
            float v = 0.0f;
            if (r < nr) {
                const float p0 = a.qss[q0 + r], p1 = a.qss[(size_t)a.qnpos + q0 + r], p2 = a.qss[2 * (size_t)a.qnpos + q0 + r];
                v = p0 * a.ssss[(int)(p0 * 9.999f) * 30 + g];
                v = fmaf(p1, a.ssss[(10 + (int)(p1 * 9.999f)) * 30 + g], v);
                v = fmaf(p2, a.ssss[(20 + (int)(p2 * 9.999f)) * 30 + g], v);
                if (g == 0) qh[r] = p2 + 0.1f;
            } else if (g == 0) qh[r] = 0.0f;
            qt[g][r] = v;
        }
    }
    for (int i = threadIdx.x; i < 20 * SC_ROWS; i += blockDim.x) {
        const int k = i / SC_ROWS, r = i % SC_ROWS;
        qf[k][r] = r < nr ? a.qtrg[(size_t)k * a.qnpos + q0 + r] : 0.0f;
    }
    if (threadIdx.x < 20)
        w[threadIdx.x] = 1.0f / (0.5f * (a.qbkg[(size_t)threadIdx.x * a.qnprof + P.q] + a.dbkg[(size_t)threadIdx.x * a.dnprof + P.p]));
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    float* out = a.S + P.soff + (int64_t)r0 * P.L2;
    /* units of 16 rows x 64 columns, dealt to the waves */
    const int nblk = (P.L2 + 63) / 64, nun = nblk * ((nr + 15) / 16);
    for (int u = wv; u < nun; u += 4) {
        const int half = u >= nblk ? 1 : 0;
        const int c = 64 * (u - half * nblk) + lane;
        const bool ok = c < P.L2;
        const int64_t col = d0 + (ok ? c : 0);
        float dw[20], pj[3], dh = 0.0f;
        int it[3] = {0, 0, 0};
#pragma unroll
        for (int k = 0; k < 20; k++) dw[k] = a.dtrg[(size_t)k * a.dnpos + col] * w[k];
        if (ss_on) {
#pragma unroll
            for (int j = 0; j < 3; j++) {
                pj[j] = a.dss[(size_t)j * a.dnpos + col];
                it[j] = 10 * j + (int)(pj[j] * 9.999f);
            }
            dh = (pj[2] + 0.1f) * 0.1111111f;
        }
        const int re = min(nr, 16 * half + 16);
        for (int r = 16 * half; r < re; r += 4) {
            float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f}, sc[4];
#pragma unroll
            for (int k = 0; k < 20; k++) {
                const float4 q = *(const float4*)&qf[k][r];
                acc[0] = fmaf(q.x, dw[k], acc[0]); acc[1] = fmaf(q.y, dw[k], acc[1]);
                acc[2] = fmaf(q.z, dw[k], acc[2]); acc[3] = fmaf(q.w, dw[k], acc[3]);
            }
            c2_logf_clamped_n<4>(acc, sc);
#pragma unroll
            for (int n = 0; n < 4; n++) sc[n] = sc[n] - a.shift;
            if (ss_on) {
                const float4 t0 = *(const float4*)&qt[it[0]][r], t1 = *(const float4*)&qt[it[1]][r],
                             t2 = *(const float4*)&qt[it[2]][r], h4 = *(const float4*)&qh[r];
                const float x0[4] = {t0.x, t0.y, t0.z, t0.w}, x1[4] = {t1.x, t1.y, t1.z, t1.w},
                            x2[4] = {t2.x, t2.y, t2.z, t2.w}, xh[4] = {h4.x, h4.y, h4.z, h4.w};
#pragma unroll
                for (int n = 0; n < 4; n++) {
                    float ss = x0[n] * pj[0];
                    ss = fmaf(x1[n], pj[1], ss);
                    ss = fmaf(x2[n], pj[2], ss);
                    ss = fmaf(xh[n], dh, ss);
                    sc[n] += (ss - 0.05f) * a.ssswgt;
                }
            }
            if (ok) {
                float* o = out + (int64_t)r * P.L2 + c;
#pragma unroll
                for (int n = 0; n < 4; n++)
                    if (r + n < re) o[(int64_t)n * P.L2] = sc[n];
            }
        }
    }
}

}  // namespace

int64_t c2_sdp_ckpt_floats() { return CKPT; }
int64_t c2_sdp_group_floats() { return QUAD; }

hipError_t c2_launch_sdp(const SdpArgs& a, bool adjoint, int groups, int nw, int64_t xoff, int64_t xn, hipStream_t stream)
{
    (void)hipGetLastError();   /* the status read after the launches is theirs alone */
    if (a.npairs <= 0) return hipSuccess;
    if (groups < 1 || nw < 1 || nw > C2_SDP_BAND) return hipErrorInvalidValue;
    if (a.K < 0 || (a.K > 0 && (a.K < 16 || 64 % a.K != 0))) return hipErrorInvalidValue;
    if (a.head) {
        const int64_t blocks = std::max<int64_t>(1, std::min<int64_t>(2048, (xn + 255) / 256));
        hipLaunchKernelGGL(k_sdp_begin, dim3((unsigned)blocks), dim3(256), 0, stream, (uint32_t*)a.head,
                           (uint32_t*)(a.ws + xoff), xn);
    }
    if (!adjoint) hipLaunchKernelGGL(k_sdp_fwd, dim3(groups), dim3(64 * nw), 0, stream, a);
    else if (a.K > 0) hipLaunchKernelGGL((k_sdp_adj<true>), dim3(groups), dim3(64 * nw), 0, stream, a);
    else hipLaunchKernelGGL((k_sdp_adj<false>), dim3(groups), dim3(64 * nw), 0, stream, a);
    if (a.head)
        hipLaunchKernelGGL(k_sdp_sums, dim3((unsigned)((a.npairs + 255) / 256)), dim3(256), 0, stream, a, adjoint ? 1 : 0);
    return hipGetLastError();
}

int c2_sdp_score_rows() { return SC_ROWS; }

hipError_t c2_launch_sdp_scores(const SdpScoreArgs& a, int nitems, hipStream_t stream)
{
    (void)hipGetLastError();   /* the status read after the launches is theirs alone */
    if (nitems <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_sdp_scores, dim3(nitems), dim3(256), 0, stream, a);
    return hipGetLastError();
}
