// Block line relaxation with the line solves parallel inside each line (option lr_solve = 1,
// and the only form for FP32-LHS and for the zebra line order).
//
// The reference (ref/lrelax.f:225-561, ref/btlu3.f:52-624) solves each line's 3x3
// block-tridiagonal system by block Thomas: the factorisation B_i = b_i - a_i C_(i-1),
// C_i = B_i^-1 c_i, then y_i = B_i^-1 (r_i - a_i y_(i-1)) forward and x_i = y_i - C_i x_(i+1)
// backward.  The factorisation does not depend on the right-hand side, so it is done once per
// direction for all lines at once (k_lr_factor); it also forms
// M_i = -B_i^-1 a_i, so that both substitutions are affine recurrences,
//     y_i = M_i y_(i-1) + B_i^-1 r_i,        x_i = (-C_i) x_(i+1) + y_i,
// and each is a prefix scan of affine maps (3x3 matrix, 3-vector) along the line.  One
// workgroup solves one line: every thread composes the maps of its P consecutive points,
// the waves scan their lanes' maps with shuffles (six doubling steps), the waves' totals are
// chained through LDS (a 3x3 matrix-vector product per wave), and every thread re-applies
// its own maps from the value entering its segment.  Two barriers per line.
//
// Lines keep the reference's Gauss-Seidel order (one workgroup walks them, line l reading
// the dq of line l-1 that it has just produced -- kept in registers, since a thread owns
// the same points of every line), or the zebra order (every line of one parity at once,
// one workgroup per line).  The arithmetic is reassociated, so results agree with the
// reference to rounding, not bit for bit.
//
// Operands are staged line-major: point i of line l at l*len + i in every plane, which is
// the natural layout for xi lines; for eta lines the factor kernel writes its planes
// transposed and s, dq are transposed around the eta sweeps.  The SA's line relaxation
// (lreltur / scatri, ref/lreltur.f:52-359) uses the same sweep with 1x1 blocks.
#include "smac_dev.h"
#include "smac_kernels.h"

// This file's arithmetic is reassociated anyway, so multiply-adds may fuse here (the library
// is otherwise built without contraction, which keeps the reference-order paths bit-exact).
#pragma clang fp contract(fast)

namespace smac {

// operand planes per point: factored diagonal (B, or 1/b for the scalar system), M, -C,
// the block to the previous line and the block to the next line
template <int NEQ> constexpr int lr_planes() { return 5 * NEQ * NEQ; }

template <typename T, int NEQ>
struct Aff {
    T m[NEQ * NEQ];   // entry (r, c) at r + NEQ*c
    T v[NEQ];
};

// a <- a o b (b applied first)
template <typename T, int NEQ>
SMAC_DEV void aff_after(Aff<T, NEQ> &a, const Aff<T, NEQ> &b)
{
    Aff<T, NEQ> o;
#pragma unroll
    for (int r = 0; r < NEQ; ++r) {
#pragma unroll
        for (int c = 0; c < NEQ; ++c) {
            T acc = a.m[r] * b.m[NEQ * c];
#pragma unroll
            for (int k = 1; k < NEQ; ++k) acc = acc + a.m[r + NEQ * k] * b.m[k + NEQ * c];
            o.m[r + NEQ * c] = acc;
        }
        T acc = a.v[r];
#pragma unroll
        for (int k = 0; k < NEQ; ++k) acc = acc + a.m[r + NEQ * k] * b.v[k];
        o.v[r] = acc;
    }
    a = o;
}

template <typename T, int NEQ>
SMAC_DEV void aff_apply(const T *m, const T *v, const T *x, T *out)
{
#pragma unroll
    for (int r = 0; r < NEQ; ++r) {
        T acc = v[r];
#pragma unroll
        for (int k = 0; k < NEQ; ++k) acc = acc + m[r + NEQ * k] * x[k];
        out[r] = acc;
    }
}

// another lane's value by a DPP move; zero where the move has no source lane
template <int CTRL> SMAC_DEV float dpp_of(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL,
                                                                 0xf, 0xf, true));
}
template <int CTRL> SMAC_DEV double dpp_of(double v)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                            (unsigned long long)(unsigned)lo));
}

// the value OFF lanes below (UP) or above; lanes that have none get anything.  One lane is a
// DPP move and half a wave a swap of halves; the distances between go through the LDS crossbar,
// whose latency of about 120 cycles a wave alone on its SIMD has nothing to fill with.
template <int OFF, bool UP> SMAC_DEV int lane_shift(int v, int lane)
{
    if constexpr (OFF == 1)
        return __builtin_amdgcn_update_dpp(0, v, UP ? 0x138 : 0x130, 0xf, 0xf, true);
    else if constexpr (OFF == 32)
        return __builtin_amdgcn_permlane32_swap(v, v, false, false)[UP ? 0 : 1];
    else
        return __builtin_amdgcn_ds_bpermute(4 * (UP ? lane - OFF : lane + OFF), v);
}
template <int OFF, bool UP> SMAC_DEV float lane_shift(float v, int lane)
{
    return __builtin_bit_cast(float, lane_shift<OFF, UP>(__builtin_bit_cast(int, v), lane));
}
template <int OFF, bool UP> SMAC_DEV double lane_shift(double v, int lane)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)lane_shift<OFF, UP>((int)(unsigned)u, lane);
    const unsigned hi = (unsigned)lane_shift<OFF, UP>((int)(unsigned)(u >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// ------------------------------------------------------------------------------------------
// factorisation: the block Thomas recurrence of btlu3j / btlu3k (ref/btlu3.f:52-624) and of
// scatri (ref/lreltur.f:337-359), for every line of both directions in one launch:
//     T_i = b_i - a_i C_(i-1),   C_i = T_i^-1 c_i            (a_0 = 0, c_(len-1) = 0)
// Lane u of a group of CH lanes holds point c0+u of a line (the whole wave, or one of the four
// 16-lane DPP rows of a wave that takes four lines).  In every step every lane forms T, adj(T),
// det(T) and C of its own point from the C that the lane before it held (a DPP shift; the
// group's first lane takes the one left by the chunk before): after u+1 steps lane u's value is
// that of the recurrence, and forming it again in later steps leaves it as it is.  So a chunk
// of CH points takes CH steps of about 110 instructions in registers alone, with no LDS access,
// broadcast or capture, and T^-1 and M = -T^-1 a follow from what the lanes hold at its end.
// The bound is the issue of those instructions, one per 5 cycles for a wave alone on its SIMD,
// over half the longest line.  Broadcasting every point's blocks through LDS to a recurrence
// that all lanes form alike took 238 us at 945x241 in FP64 and 116 at 705x173 in FP32; this
// takes 152 and 91 (reference-order FP32 945x241, whole lines: 287 and 255).
// (The reference keeps T_i as LU factors; the explicit inverse makes the sweeps' T_i^-1 r_i a
// parallel product.)  The blocks to the neighbouring lines pass through to the operand planes.

// 1/x: the hardware reciprocal refined by Newton-Raphson steps r <- r + r (1 - x r), each of
// which doubles the number of correct bits (two for FP64, one for FP32)
SMAC_DEV double rcp_nr(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    double e = 1.0 - x * r;
    r = r + r * e;
    e = 1.0 - x * r;
    return r + r * e;
}
SMAC_DEV float rcp_nr(float x)
{
    const float r = __builtin_amdgcn_rcpf(x);
    return r + r * (1.0f - x * r);
}

// adj(T) (column-major, entry (r, c) at r + 3c) and det(T) of a 3x3 T
template <typename T>
SMAC_DEV T adj3(const T t[9], T adj[9])
{
    adj[0] = t[4] * t[8] - t[7] * t[5];
    adj[1] = t[7] * t[2] - t[1] * t[8];
    adj[2] = t[1] * t[5] - t[4] * t[2];
    adj[3] = t[6] * t[5] - t[3] * t[8];
    adj[4] = t[0] * t[8] - t[6] * t[2];
    adj[5] = t[3] * t[2] - t[0] * t[5];
    adj[6] = t[3] * t[7] - t[6] * t[4];
    adj[7] = t[6] * t[1] - t[0] * t[7];
    adj[8] = t[0] * t[4] - t[3] * t[1];
    return t[0] * adj[0] + t[3] * adj[1] + t[6] * adj[2];
}

// out = x y (NEQ x NEQ, column-major)
template <typename T, int NEQ>
SMAC_DEV void mm(const T *x, const T *y, T *out)
{
#pragma unroll
    for (int r = 0; r < NEQ; ++r)
#pragma unroll
        for (int c = 0; c < NEQ; ++c) {
            T acc = x[r] * y[NEQ * c];
#pragma unroll
            for (int k = 1; k < NEQ; ++k) acc = acc + x[r + NEQ * k] * y[k + NEQ * c];
            out[r + NEQ * c] = acc;
        }
}

// The line is split at m = len/2 and eliminated from both ends at once (a twisted
// factorisation): wave 0 runs the recurrence forward over points 0..m-1,
//     T_i = b_i - a_i C_(i-1),   C_i = T_i^-1 c_i,      M_i = -T_i^-1 a_i,
// wave 1 runs it backward over points len-1..m+1,
//     T_i = b_i - c_i D_(i+1),   D_i = T_i^-1 a_i,      M_i = -T_i^-1 c_i,
// and the middle point takes both: T_m = b_m - a_m C_(m-1) - c_m D_(m+1), with
// Ma = -T_m^-1 a_m and Mc = -T_m^-1 c_m.  Each half's chain is half the line.  Planes per
// point: T^-1; M (Ma at m); -C or -D (Mc at m); the blocks to the previous and next line.  In
// the planes a line's points stand in the order of the sweeps' scans: the first half, the
// second from its end, the middle point.
// A workgroup takes LPW lines (1 or 4), wave 0 their first halves and wave 1 their second.
constexpr int FW = 64;

// t -= x C, and for T = t - x C:  det(T) and adj(T) (T^-1 = adj / det)
template <typename LT, int NEQ>
SMAC_DEV void lr_less(const LT *x, LT *t, const LT *C)
{
#pragma unroll
    for (int cc = 0; cc < NEQ; ++cc)
#pragma unroll
        for (int r = 0; r < NEQ; ++r)
#pragma unroll
            for (int k = 0; k < NEQ; ++k)
                t[r + NEQ * cc] = t[r + NEQ * cc] - x[r + NEQ * k] * C[k + NEQ * cc];
}
template <typename LT, int NEQ>
SMAC_DEV LT lr_pivot(const LT *x, LT *t, const LT *C, LT *ad)
{
    lr_less<LT, NEQ>(x, t, C);
    if constexpr (NEQ == 3) return adj3(t, ad);
    ad[0] = (LT)1;
    return t[0];
}

template <typename LT, int NEQ, int LPW>
SMAC_DEV void lr_factor(const Dims &d, bool eta, int grp, int twist, const LT *__restrict__ btc,
                        const LT *__restrict__ lm, const LT *__restrict__ lp,
                        const LT *__restrict__ om, const LT *__restrict__ opn,
                        LT *__restrict__ out, LT (*edge)[4][NEQ * NEQ])
{
    constexpr int NB = NEQ * NEQ, CH = FW / LPW;
    constexpr int SHR = LPW == 1 ? 0x138 : 0x111, ROR = LPW == 1 ? 0x13c : 0x121;   // wave / row
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, u = lane % CH, row = lane / CH;
    const int nline = eta ? d.jm : d.km, len = eta ? d.km : d.jm;
    const int l = grp * LPW + row;
    const bool on = l < nline;
    // twist = 0: the plain (one-sided) factorisation, forward over the whole line (wave 0;
    // launched with one wave)
    const int mid = twist ? len / 2 : len;
    const long N = d.N;
    const long stride = eta ? d.jm : 1, base = eta ? (long)l : (long)l * d.jm;
    // wave 0 walks points 0, 1, .., mid-1; wave 1 walks len-1, len-2, .., mid+1
    const bool fwd = wv == 0;
    const int first = fwd ? 0 : len - 1, count = fwd ? mid : (len - 1 - mid > 0 ? len - 1 - mid : 0),
              step = fwd ? 1 : -1;
    // forward: the carried side is a (times C of the point before), the solved side c;
    // backward the other way round
    const LT *carried = fwd ? lm : lp, *solved = fwd ? lp : lm;
    struct Pt { LT car[NB], b[NB], sol[NB]; } cur, nxt;
    auto load = [&](Pt &t, int c0) {
        const int v = c0 + u;
        if (on && v < count) {
            const int i = first + step * v;
            const long p = base + stride * i;
            const bool has_a = i > 0, has_c = i < len - 1;
            const bool has_car = fwd ? has_a : has_c, has_sol = fwd ? has_c : has_a;
#pragma unroll
            for (int e = 0; e < NB; ++e) {
                t.b[e] = btc[e * N + p];
                t.car[e] = has_car ? carried[e * N + p] : (LT)0;
                t.sol[e] = has_sol ? solved[e * N + p] : (LT)0;
            }
        }
    };
    LT C[NB], carry[NB], ad[NB], rd = (LT)0;
#pragma unroll
    for (int e = 0; e < NB; ++e) {
        C[e] = carry[e] = ad[e] = (LT)0;
        cur.b[e] = cur.car[e] = cur.sol[e] = nxt.b[e] = nxt.car[e] = nxt.sol[e] = (LT)0;
    }
    load(cur, 0);
    for (int c0 = 0; c0 < count; c0 += CH) {
        const int v = c0 + u;
        const bool act = on && v < count;
        const long p = base + stride * (first + step * v);
        const long o = (long)l * len + (fwd ? v : mid + v);
        if (c0 + CH < count) load(nxt, c0 + CH);
        LT rom[NB], rop[NB];
        if (act) {
#pragma unroll
            for (int e = 0; e < NB; ++e) {
                rom[e] = om[e * N + p];
                rop[e] = opn[e * N + p];
            }
        }
        const int nv = count - c0 < CH ? count - c0 : CH;
        // the group's first lane takes its product with the carried value here, and nothing
        // from a neighbour in the steps
        LT car[NB];
        {
            LT t[NB];
#pragma unroll
            for (int e = 0; e < NB; ++e) t[e] = cur.b[e];
            lr_less<LT, NEQ>(cur.car, t, carry);
#pragma unroll
            for (int e = 0; e < NB; ++e) {
                cur.b[e] = u == 0 ? t[e] : cur.b[e];
                car[e] = u == 0 ? (LT)0 : cur.car[e];
            }
        }
        for (int s = 0; s < nv; ++s) {
            LT x[NB], t[NB], ac[NB];
#pragma unroll
            for (int e = 0; e < NB; ++e) {
                x[e] = dpp_of<SHR>(C[e]);
                t[e] = cur.b[e];
            }
            const LT det = lr_pivot<LT, NEQ>(car, t, x, ad);
            mm<LT, NEQ>(ad, cur.sol, ac);
            rd = rcp_nr(det);
#pragma unroll
            for (int e = 0; e < NB; ++e) C[e] = ac[e] * rd;
        }
        if (act) {
            LT bi[NB], m[NB];
#pragma unroll
            for (int e = 0; e < NB; ++e) bi[e] = ad[e] * rd;
            mm<LT, NEQ>(bi, cur.car, m);
#pragma unroll
            for (int e = 0; e < NB; ++e) {
                out[e * N + o] = bi[e];
                out[(NB + e) * N + o] = -m[e];
                out[(2 * NB + e) * N + o] = -C[e];
                out[(3 * NB + e) * N + o] = rom[e];
                out[(4 * NB + e) * N + o] = rop[e];
            }
        }
        if (c0 + CH >= count) {
            if (u == nv - 1) {
#pragma unroll
                for (int e = 0; e < NB; ++e) edge[wv][row][e] = C[e];   // C_(m-1) / D_(m+1)
            }
        } else {
#pragma unroll
            for (int e = 0; e < NB; ++e) carry[e] = dpp_of<ROR>(C[e]);
            cur = nxt;
        }
    }
    if (!twist) return;
    if (count == 0 && u == 0) {
#pragma unroll
        for (int e = 0; e < NB; ++e) edge[wv][row][e] = (LT)0;
    }
    __syncthreads();
    // the middle point
    if (wv == 0 && u == 0 && on) {
        const long p = base + stride * mid, o = (long)l * len + len - 1;
        LT a[NB], b[NB], c[NB], t[NB], am[NB], w[NB];
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            b[e] = btc[e * N + p];
            a[e] = mid > 0 ? lm[e * N + p] : (LT)0;
            c[e] = mid < len - 1 ? lp[e * N + p] : (LT)0;
            out[(3 * NB + e) * N + o] = om[e * N + p];
            out[(4 * NB + e) * N + o] = opn[e * N + p];
            t[e] = b[e];
        }
        lr_pivot<LT, NEQ>(a, t, edge[0][row], am);              // b - a C_(m-1)
        const LT det = lr_pivot<LT, NEQ>(c, t, edge[1][row], am);   // - c D_(m+1)
        const LT rm = rcp_nr(det);
        LT bi[NB];
#pragma unroll
        for (int e = 0; e < NB; ++e) bi[e] = am[e] * rm;
        mm<LT, NEQ>(bi, a, w);
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            out[e * N + o] = bi[e];
            out[(NB + e) * N + o] = -w[e];
        }
        mm<LT, NEQ>(bi, c, w);
#pragma unroll
        for (int e = 0; e < NB; ++e) out[(2 * NB + e) * N + o] = -w[e];
    }
}

// workgroups [0, nx) take the xi lines (k = const: contiguous along the line), the rest the eta
// lines (j = const: stride jm); lpx, lpe: lines per workgroup of each
template <typename LT, int NEQ>
__global__ void __launch_bounds__(2 * FW)
k_lr_factor(Dims d, int nx, int lpx, int lpe, int twist, const LT *__restrict__ btc,
            const LT *__restrict__ bjm, const LT *__restrict__ bjp, const LT *__restrict__ bkm,
            const LT *__restrict__ bkp, LT *__restrict__ opx, LT *__restrict__ ope)
{
    __shared__ LT edge[2][4][NEQ * NEQ];   // per half and line of the workgroup
    if ((int)blockIdx.x < nx) {
        // the xi lines are the longer chains: their waves win issue slots on a shared SIMD
        __builtin_amdgcn_s_setprio(2);
        if (lpx == 1)
            lr_factor<LT, NEQ, 1>(d, false, (int)blockIdx.x, twist, btc, bjm, bjp, bkm, bkp, opx, edge);
        else
            lr_factor<LT, NEQ, 4>(d, false, (int)blockIdx.x, twist, btc, bjm, bjp, bkm, bkp, opx, edge);
        return;
    }
    // eta lines: a point's planes are read by lanes jm apart, and the lines of neighbouring j
    // share those cache lines; workgroups reach the 8 XCDs round-robin, so each XCD takes a
    // contiguous run of j (its own L2 then holds the shared lines)
    const int t = (int)blockIdx.x - nx, ne = (int)gridDim.x - nx;
    const int r = t % 8, q = ne / 8, rem = ne % 8;
    const int g = r * q + (r < rem ? r : rem) + t / 8;
    if (lpe == 1)
        lr_factor<LT, NEQ, 1>(d, true, g, twist, btc, bkm, bkp, bjm, bjp, ope, edge);
    else
        lr_factor<LT, NEQ, 4>(d, true, g, twist, btc, bkm, bkp, bjm, bjp, ope, edge);
}

// Lines per workgroup.  One where the direction's waves (two per line when twisted) find a SIMD
// each: a chunk of 64 points loads and stores coalesced and pays its ends once per 64 steps.
// Four where they do not: two waves on a SIMD halve each other's rate, and four lines in one
// wave take the steps of one.  Twisted FP64 945x241 (241 xi lines, 945 eta lines): one line
// everywhere 212 us, four everywhere 202, the xi lines singly and the eta lines by four 160;
// FP32 705x173 101, 109, 92.  Below the line one per workgroup stays the better: 203x47 FP64
// 36 us against 42, the plain FP32 factorisation of 945x241 255 against 289.
static int lines_per_group(int nline, bool twist) { return nline * (twist ? 2 : 1) <= 1024 ? 1 : 4; }

// ------------------------------------------------------------------------------------------
// the sweep: lines count of them, line l = (first + idx*step) mod nline, one workgroup per line
// (lines of one colour); k_lr_walk below takes them in order in one workgroup.
// s, dq: NEQ planes, line-major; op: the factor kernel's planes.  assign: dq = x (the SA's
// lreltur); otherwise dq += underr (x - dq) (ref/lrelax.f:377-381).
//
// The solve follows the twisted factorisation (mid = len/2):
//   phase 1  y_i = M_i y_(i-1) + T_i^-1 r_i  forward over i < mid, and
//            z_i = M_i z_(i+1) + T_i^-1 r_i  backward over i > mid, both scans at once
//            (each point's map is the identity in the scan of the other half); then
//            x_mid = T^-1 r + Ma y_(mid-1) + Mc z_(mid+1) in the thread owning mid;
//   phase 2  x_i = -C_i x_(i+1) + y_i  backward over i < mid, and
//            x_i = -D_i x_(i-1) + z_i  forward over i > mid, the point mid entering both
//            scans as the constant map x_mid.
//
// What bounds a sweep of one colour is how fast the few workgroups (121 of 945 points) can draw
// their operands, then the latency of the scan's exchanges.  With every load in flight before
// the first wait, pairs of points in one load, the scan without branches, and its distances 1
// and 32 as DPP move and half-wave swap instead of crossbar reads, a 945x241 FP64 xi colour
// takes 18.6 us (28.6 before) and an eta colour 16.4 (17.9); FP32 at 705x173 11.7 (14.1) and 9.2
// (10.1).

// one doubling step: the lane's map after that of OFF lanes before
template <typename AT, int NEQ, bool FWD, int OFF>
SMAC_DEV void scan_level(Aff<AT, NEQ> &agg, int lane)
{
    Aff<AT, NEQ> o, n = agg;
#pragma unroll
    for (int e = 0; e < NEQ * NEQ; ++e) o.m[e] = lane_shift<OFF, FWD>(agg.m[e], lane);
#pragma unroll
    for (int e = 0; e < NEQ; ++e) o.v[e] = lane_shift<OFF, FWD>(agg.v[e], lane);
    aff_after(n, o);
    const bool has = FWD ? lane >= OFF : lane + OFF < 64;
#pragma unroll
    for (int e = 0; e < NEQ * NEQ; ++e) agg.m[e] = has ? n.m[e] : agg.m[e];
#pragma unroll
    for (int e = 0; e < NEQ; ++e) agg.v[e] = has ? n.v[e] : agg.v[e];
}

// the value entering wave wv: the maps of the waves before it, one after the other, from zero.
// Their totals are read from LDS four at a time ahead of the products, where the registers
// hold them (8 waves of FP64 3x3 maps: one at a time).
template <typename AT, int NEQ, int NW, bool FWD>
SMAC_DEV void wave_entry(const AT (*tot)[NEQ * NEQ + NEQ], int wv, AT *Y)
{
    constexpr int NB = NEQ * NEQ, G = sizeof(AT) * NEQ * NW > 96 ? 1 : 4;
    const int before = __builtin_amdgcn_readfirstlane(FWD ? wv : NW - 1 - wv);
#pragma unroll
    for (int n = 0; n < NEQ; ++n) Y[n] = (AT)0;
#pragma unroll
    for (int k0 = 0; k0 < NW - 1; k0 += G) {
        if (k0 >= before) break;
        AT a[G][NB + NEQ];
#pragma unroll
        for (int i = 0; i < G; ++i)
            if (k0 + i < NW - 1)
#pragma unroll
                for (int e = 0; e < NB + NEQ; ++e)
                    a[i][e] = tot[FWD ? k0 + i : NW - 1 - k0 - i][e];
#pragma unroll
        for (int i = 0; i < G; ++i)
            if (k0 + i < NW - 1 && k0 + i < before) {
                AT nY[NEQ];
                aff_apply<AT, NEQ>(a[i], a[i] + NB, Y, nY);
#pragma unroll
                for (int n = 0; n < NEQ; ++n) Y[n] = nY[n];
            }
    }
}

// one scan of the thread's PP points along the line (FWD: ascending, else descending) with
// the value 0 entering the line: get(u, a) gives point u's map, put(u, x) receives the value
// after it.  tot: the waves' totals in LDS (the caller synchronises before it is written
// again).
template <typename AT, int NEQ, int NT, int PP, bool FWD, class Get, class Put>
SMAC_DEV void line_scan(Get get, Put put, AT (*tot)[NEQ * NEQ + NEQ], int lane, int wv)
{
    constexpr int NB = NEQ * NEQ, NW = NT / 64;
    Aff<AT, NEQ> agg;
#pragma unroll
    for (int k = 0; k < PP; ++k) {
        const int u = FWD ? k : PP - 1 - k;
        Aff<AT, NEQ> a;
        get(u, a);
        if (k == 0) agg = a;
        else {
            aff_after(a, agg);
            agg = a;
        }
    }
    scan_level<AT, NEQ, FWD, 1>(agg, lane);
    scan_level<AT, NEQ, FWD, 2>(agg, lane);
    scan_level<AT, NEQ, FWD, 4>(agg, lane);
    scan_level<AT, NEQ, FWD, 8>(agg, lane);
    scan_level<AT, NEQ, FWD, 16>(agg, lane);
    scan_level<AT, NEQ, FWD, 32>(agg, lane);
    if (lane == (FWD ? 63 : 0)) {
#pragma unroll
        for (int e = 0; e < NB; ++e) tot[wv][e] = agg.m[e];
#pragma unroll
        for (int n = 0; n < NEQ; ++n) tot[wv][NB + n] = agg.v[n];
    }
    __syncthreads();
    // the value entering this wave, then this thread
    AT Y[NEQ];
    wave_entry<AT, NEQ, NW, FWD>(tot, wv, Y);
    AT ye[NEQ], cur[NEQ];
    aff_apply<AT, NEQ>(agg.m, agg.v, Y, ye);
#pragma unroll
    for (int n = 0; n < NEQ; ++n) {
        const AT nb = lane_shift<1, FWD>(ye[n], lane);
        cur[n] = lane == (FWD ? 0 : 63) ? Y[n] : nb;
    }
#pragma unroll
    for (int k = 0; k < PP; ++k) {
        const int u = FWD ? k : PP - 1 - k;
        Aff<AT, NEQ> a;
        get(u, a);
        AT nx[NEQ];
        aff_apply<AT, NEQ>(a.m, a.v, cur, nx);
#pragma unroll
        for (int n = 0; n < NEQ; ++n) cur[n] = nx[n];
        put(u, cur);
    }
}

template <typename AT, int NEQ>
SMAC_DEV void aff_identity(Aff<AT, NEQ> &a)
{
#pragma unroll
    for (int r = 0; r < NEQ; ++r) {
#pragma unroll
        for (int c = 0; c < NEQ; ++c) a.m[r + NEQ * c] = r == c ? (AT)1 : (AT)0;
        a.v[r] = (AT)0;
    }
}

// a thread's PP points of NB planes from p on, a pair in one load (of element alignment): with
// an odd length the last pair reaches one element past the line, which nothing uses; past the
// last line of the last plane lie the operands' 256 bytes of padding
template <typename T, int NB, int PP>
SMAC_DEV void load_planes(T (&x)[PP][NB], const T *p, long N)
{
    static_assert(PP == 1 || PP == 2, "one point or a pair");
    typedef T Pair __attribute__((ext_vector_type(2), aligned(sizeof(T))));
#pragma unroll
    for (int e = 0; e < NB; ++e) {
        if constexpr (PP == 2) {
            const Pair y = *(const Pair *)(p + e * N);
            x[0][e] = y.x;
            x[1][e] = y.y;
        } else {
            x[0][e] = p[e * N];
        }
    }
}

// acc += block x, where there is such a line
template <typename LT, int NEQ>
SMAC_DEV void lr_terms(double *acc, bool has, const LT *b, const double *x)
{
#pragma unroll
    for (int m = 0; m < NEQ; ++m) {
        double t = acc[m];
#pragma unroll
        for (int k = 0; k < NEQ; ++k) t += (double)b[m + NEQ * k] * x[k];
        acc[m] = has ? t : acc[m];
    }
}

// A colour step of the transposed sweeps (TRANS; see below): dq is z, s is not read
struct LrTStep {
    double *a, *sbar;
    double w;
    int spread;   // the other colour's z belongs to the step before: a takes its terms first
    int begin;    // the colour's first step: sbar starts from zero
};

template <typename LT, int NEQ, int NT, int PP, bool TWIST, bool TRANS>
__global__ void __launch_bounds__(NT)
k_lr_sweep(int nline, int len, long N, int count, int first, int step, double underr,
           int assign, double *__restrict__ dq, const double *__restrict__ s,
           const LT *__restrict__ op, LrTStep ts)
{
    using AT = LT;
    constexpr int NB = NEQ * NEQ, NW = NT / 64;
    __shared__ AT lf[NW][NB + NEQ], lb[NW][NB + NEQ];
    __shared__ AT xch[2][NEQ];   // twisted: y_(mid-1) to the middle point, x_mid back
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    // The plain factorisation: the forward half is the whole line.  The twisted one: the
    // scans run over the line's points renumbered v = 0..len-1 as the first half in order
    // (i = v < mid), the second half reversed (i = len - 1 - (v - mid)) and the middle point
    // last, so that each phase is one scan: phase 1 forward, restarted where the second half
    // begins (i = len - 1, whose map ignores what comes before it), and phase 2 backward from
    // the middle point, the first half restarted from x_mid.
    const int mid = TWIST ? len / 2 : len;
    auto phys = [&](int v) { return (!TWIST || v < mid) ? v : (v < len - 1 ? len - 1 - v + mid : mid); };
    const LT *pB = op, *pM = op + NB * N, *pC = op + 2 * NB * N, *pOm = op + 3 * NB * N,
             *pOp = op + 4 * NB * N;
    // point u's place in the natural planes
    auto nat = [&](int l, int u) {
        const int v = t * PP + u;
        return (long)l * len + phys(v < len ? v : len - 1);
    };
    for (int idx = (int)blockIdx.x; idx < count; idx += (int)gridDim.x) {
        const int l = (first + idx * step) % nline;
        const bool hm = l > 0, hp = l < nline - 1;
        AT mmat[PP][NB];               // M (Ma at mid)
        AT bv[PP][NEQ];                // T^-1 r
        AT w[PP][NEQ];                 // y (i < mid) or z (i > mid); z_(mid+1), then x_mid, at
                                       // the middle point; then x
        // ---- this thread's points: T^-1 r, M, -C / -D.  Past the line's end (and beyond the
        // first and last line) stand in-range addresses whose values are not used: without
        // branches every load is in flight before the first is waited for.
        const long lo = (long)l * len + (t * PP < len ? t * PP : len - 1);
        AT bi[PP][NB];
        double r[PP][NEQ], sb[PP][NEQ];
        load_planes(bi, pB + lo, N);
        load_planes(mmat, pM + lo, N);
#pragma unroll
        for (int u = 0; u < PP; ++u)
#pragma unroll
            for (int n = 0; n < NEQ; ++n) {
                r[u][n] = (TRANS ? ts.a : s)[n * N + nat(l, u)];
                if constexpr (TRANS) sb[u][n] = ts.begin ? 0.0 : ts.sbar[n * N + nat(l, u)];
            }
        if (!TRANS || ts.spread) {
            AT om[PP][NB], op_[PP][NB];
            double xm[PP][NEQ], xp[PP][NEQ];
            load_planes(om, pOm + lo, N);
            load_planes(op_, pOp + lo, N);
#pragma unroll
            for (int u = 0; u < PP; ++u)
#pragma unroll
                for (int n = 0; n < NEQ; ++n) {
                    xm[u][n] = dq[n * N + nat(hm ? l - 1 : l, u)];
                    xp[u][n] = dq[n * N + nat(hp ? l + 1 : l, u)];
                }
            if constexpr (TRANS) {
#pragma unroll
                for (int u = 0; u < PP; ++u) {
                    double acc[NEQ] = {};
                    lr_terms<LT, NEQ>(acc, hm, om[u], xm[u]);
                    lr_terms<LT, NEQ>(acc, hp, op_[u], xp[u]);
#pragma unroll
                    for (int m = 0; m < NEQ; ++m) r[u][m] -= ts.w * acc[m];
                }
            } else {
#pragma unroll
                for (int u = 0; u < PP; ++u) {
#pragma unroll
                    for (int m = 0; m < NEQ; ++m) {
                        double b = (double)om[u][m] * xm[u][0];
#pragma unroll
                        for (int n = 1; n < NEQ; ++n) b = b + (double)om[u][m + NEQ * n] * xm[u][n];
                        r[u][m] = hm ? r[u][m] - b : r[u][m];
                    }
#pragma unroll
                    for (int m = 0; m < NEQ; ++m) {
                        double b = (double)op_[u][m] * xp[u][0];
#pragma unroll
                        for (int n = 1; n < NEQ; ++n) b = b + (double)op_[u][m + NEQ * n] * xp[u][n];
                        r[u][m] = hp ? r[u][m] - b : r[u][m];
                    }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < PP; ++u) {
            AT rr[NEQ];
#pragma unroll
            for (int n = 0; n < NEQ; ++n) rr[n] = (AT)r[u][n];
#pragma unroll
            for (int m = 0; m < NEQ; ++m) {
                AT acc = bi[u][m] * rr[0];
#pragma unroll
                for (int n = 1; n < NEQ; ++n) acc = acc + bi[u][m + NEQ * n] * rr[n];
                bv[u][m] = acc;
            }
        }
        // ---- phase 1: y forward over i < mid, z backward over i > mid, in one forward scan
        line_scan<AT, NEQ, NT, PP, true>(
            [&](int u, Aff<AT, NEQ> &a) {
                // every field written once, through selects (branches on the struct put it
                // in scratch memory): past the line and at the middle point (which passes
                // z_(mid+1) through) the identity; at the second half's first point a map
                // that ignores what comes before it
                const int v = t * PP + u;
                const bool pass = v >= len || (TWIST && v == len - 1), rst = TWIST && v == mid;
#pragma unroll
                for (int r = 0; r < NEQ; ++r) {
#pragma unroll
                    for (int c = 0; c < NEQ; ++c)
                        a.m[r + NEQ * c] = pass ? (r == c ? (AT)1 : (AT)0)
                                                : rst ? (AT)0 : mmat[u][r + NEQ * c];
                    a.v[r] = pass ? (AT)0 : bv[u][r];
                }
            },
            [&](int u, const AT *x) {
                const int v = t * PP + u;
#pragma unroll
                for (int n = 0; n < NEQ; ++n) {
                    if (v < len) w[u][n] = x[n];
                    if (TWIST && v == mid - 1) xch[0][n] = x[n];
                }
            },
            lf, lane, wv);
        // the -C / -D planes (Mc at mid), read only now: phase 1 does not need them (loaded with
        // the others, 945x241 FP64 colours take 19.2 and 17.0 us instead of 18.6 and 16.4)
        AT cm[PP][NB];
        load_planes(cm, pC + lo, N);
        __syncthreads();   // phase 1's wave totals have been read; y_(mid-1) is in xch
        // ---- the middle point: x_mid = T^-1 r + Ma y_(mid-1) + Mc z_(mid+1) (the plain
        // factorisation has none: there mid = len, past the line)
        if constexpr (TWIST) {
#pragma unroll
            for (int u = 0; u < PP; ++u)
                if (t * PP + u == len - 1) {
                    AT ymid[NEQ], zmid[NEQ];
#pragma unroll
                    for (int n = 0; n < NEQ; ++n) {
                        ymid[n] = mid > 0 ? xch[0][n] : (AT)0;
                        zmid[n] = len - 1 > mid ? w[u][n] : (AT)0;
                    }
#pragma unroll
                    for (int r = 0; r < NEQ; ++r) {
                        AT acc = bv[u][r];
#pragma unroll
                        for (int k = 0; k < NEQ; ++k)
                            acc = acc + mmat[u][r + NEQ * k] * ymid[k] + cm[u][r + NEQ * k] * zmid[k];
                        w[u][r] = acc;
                        xch[1][r] = acc;
                    }
                }
            __syncthreads();   // x_mid is in xch
        }
        // ---- phase 2: x backward over i < mid and forward over i > mid, from x_mid, in one
        // backward scan: the middle point (last) gives x_mid, the second half follows it, and
        // the first half's last point (v = mid - 1) restarts from x_mid
        line_scan<AT, NEQ, NT, PP, false>(
            [&](int u, Aff<AT, NEQ> &a) {
                // as in phase 1, every field once: past the line the identity; at the middle
                // point (0, x_mid); at the first half's last point (0, -C x_mid + y), a
                // restart from x_mid; elsewhere (-C or -D, y or z)
                const int v = t * PP + u;
                const bool past = v >= len, midp = TWIST && v == len - 1;
                const bool rst = TWIST && v == mid - 1;
                AT xm[NEQ];
#pragma unroll
                for (int k = 0; k < NEQ; ++k) xm[k] = TWIST ? xch[1][k] : (AT)0;
#pragma unroll
                for (int r = 0; r < NEQ; ++r) {
#pragma unroll
                    for (int c = 0; c < NEQ; ++c)
                        a.m[r + NEQ * c] = past ? (r == c ? (AT)1 : (AT)0)
                                                : (midp || rst) ? (AT)0 : cm[u][r + NEQ * c];
                    AT acc = w[u][r];
#pragma unroll
                    for (int k = 0; k < NEQ; ++k) acc = acc + cm[u][r + NEQ * k] * xm[k];
                    a.v[r] = past ? (AT)0 : rst ? acc : w[u][r];
                }
            },
            [&](int u, const AT *x) {
                const int v = t * PP + u;
#pragma unroll
                for (int n = 0; n < NEQ; ++n)
                    if (v < len) w[u][n] = x[n];
            },
            lb, lane, wv);
#pragma unroll
        for (int u = 0; u < PP; ++u) {
            const int v = t * PP + u;
            if (v < len) {
                const long o = (long)l * len + phys(v);
#pragma unroll
                for (int n = 0; n < NEQ; ++n) {
                    const double xd = (double)w[u][n];
                    if constexpr (TRANS) {
                        dq[n * N + o] = xd;
                        ts.sbar[n * N + o] = sb[u][n] + ts.w * xd;
                        ts.a[n * N + o] = r[u][n] * (1.0 - ts.w);
                        continue;
                    }
                    const double dold = assign ? 0.0 : dq[n * N + o];
                    const double nv = assign ? xd : dold + underr * (xd - dold);
                    dq[n * N + o] = nv;
                }
            }
        }
        __syncthreads();   // phase 2's wave totals and xch have been read before the next line
    }
}

// The reference's line order (the plain factorisation): one workgroup walks the lines, line l
// taking the dq of the line before it from registers (a thread owns the same points of every
// line) and that of the line after it, not yet updated, from memory.  The walk is one chain, bound
// by the instructions and exchanges of a line's two scans on one compute unit: the next line's
// operands are loaded during the present one's scans (AHEAD; where a line takes 1024 threads,
// their 128 registers do not hold them, and each line loads its own: FP64 1201x241 31 ms a pass
// against 53 with the spilled prefetch).  FP32-LHS 945x241: an eta line (241 points) 3.2 us, 5.7
// without prefetch and with crossbar scans, a xi line (945 points) 6.6, before 12.1; FP64 passes
// 20.0 ms, before 24.9.  (3x3 lines of up to 256 points, FP64 128, take k_lr_walk_ahead.)
template <typename LT, int NEQ, int NT, int PP>
__global__ void __launch_bounds__(NT)
k_lr_walk(int nline, int len, long N, int count, int first, int step, double underr, int assign,
          double *__restrict__ dq, const double *__restrict__ s, const LT *__restrict__ op)
{
    using AT = LT;
    constexpr int NB = NEQ * NEQ, NW = NT / 64;
    __shared__ AT lf[NW][NB + NEQ], lb[NW][NB + NEQ];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const bool up = step > 0;
    // planes of the block to the line before (near) and after (far) in the walk
    const LT *pB = op, *pM = op + NB * N, *pC = op + 2 * NB * N,
             *pNear = op + (up ? 3 : 4) * NB * N, *pFar = op + (up ? 4 : 3) * NB * N;
    LT B[PP][NB], M[PP][NB], C[PP][NB], near[PP][NB], far[PP][NB];
    double rhs[PP][NEQ], fx[PP][NEQ], own[PP][NEQ], done[PP][NEQ];
    auto line = [&](int idx) {
        const int l = (first + idx * step) % nline;
        return l < 0 ? l + nline : l;
    };
    // past the line's end in-range addresses stand, whose values nothing uses
    const int at0 = t * PP < len ? t * PP : len - 1;
    auto load = [&](LT (&x)[PP][NB], const LT *pl, int l) {
        load_planes(x, pl + (long)l * len + at0, N);
    };
    auto loadv = [&](double (&x)[PP][NEQ], const double *pl, int l) {
#pragma unroll
        for (int n = 0; n < NEQ; ++n)
#pragma unroll
            for (int u = 0; u < PP; ++u) x[u][n] = pl[n * N + (long)l * len + (t * PP + u < len ? t * PP + u : len - 1)];
    };
    // what a line needs before its scans
    auto fetch = [&](int l) {
        const int beyond = up ? l + 1 : l - 1;
        load(B, pB, l);
        load(near, pNear, l);
        load(far, pFar, l);
        loadv(rhs, s, l);
        loadv(fx, dq, beyond >= 0 && beyond < nline ? beyond : l);
    };
    constexpr bool AHEAD = NT < 1024;
    if (AHEAD) {
        fetch(line(0));
        load(M, pM, line(0));
        load(C, pC, line(0));
    }
    int lprev = -2;
    for (int idx = 0; idx < count; ++idx) {
        const int l = line(idx), ln = line(idx + 1 < count ? idx + 1 : idx);
        const bool hm = l > 0, hp = l < nline - 1;
        const bool regm = lprev == l - 1, regp = lprev == l + 1;
        AT w[PP][NEQ], bv[PP][NEQ];
        if (!AHEAD) {
            fetch(l);
            load(M, pM, l);
        }
#pragma unroll
        for (int u = 0; u < PP; ++u) {
            double r[NEQ];
#pragma unroll
            for (int n = 0; n < NEQ; ++n) r[n] = rhs[u][n];
            if (hm) {
#pragma unroll
                for (int m = 0; m < NEQ; ++m) {
                    double x[NEQ];
#pragma unroll
                    for (int n = 0; n < NEQ; ++n) x[n] = regm ? done[u][n] : fx[u][n];
                    double b = (double)(up ? near : far)[u][m] * x[0];
#pragma unroll
                    for (int n = 1; n < NEQ; ++n)
                        b = b + (double)(up ? near : far)[u][m + NEQ * n] * x[n];
                    r[m] = r[m] - b;
                }
            }
            if (hp) {
#pragma unroll
                for (int m = 0; m < NEQ; ++m) {
                    double x[NEQ];
#pragma unroll
                    for (int n = 0; n < NEQ; ++n) x[n] = regp ? done[u][n] : fx[u][n];
                    double b = (double)(up ? far : near)[u][m] * x[0];
#pragma unroll
                    for (int n = 1; n < NEQ; ++n)
                        b = b + (double)(up ? far : near)[u][m + NEQ * n] * x[n];
                    r[m] = r[m] - b;
                }
            }
            AT rr[NEQ];
#pragma unroll
            for (int n = 0; n < NEQ; ++n) rr[n] = (AT)r[n];
#pragma unroll
            for (int m = 0; m < NEQ; ++m) {
                AT acc = B[u][m] * rr[0];
#pragma unroll
                for (int n = 1; n < NEQ; ++n) acc = acc + B[u][m + NEQ * n] * rr[n];
                bv[u][m] = acc;
            }
        }
        loadv(own, dq, l);
        if (AHEAD) fetch(ln);
        line_scan<AT, NEQ, NT, PP, true>(
            [&](int u, Aff<AT, NEQ> &a) {
                const bool pass = t * PP + u >= len;
#pragma unroll
                for (int r = 0; r < NEQ; ++r) {
#pragma unroll
                    for (int c = 0; c < NEQ; ++c)
                        a.m[r + NEQ * c] = pass ? (r == c ? (AT)1 : (AT)0) : M[u][r + NEQ * c];
                    a.v[r] = pass ? (AT)0 : bv[u][r];
                }
            },
            [&](int u, const AT *x) {
#pragma unroll
                for (int n = 0; n < NEQ; ++n) w[u][n] = x[n];
            },
            lf, lane, wv);
        if (AHEAD) load(M, pM, ln);
        else load(C, pC, l);
        line_scan<AT, NEQ, NT, PP, false>(
            [&](int u, Aff<AT, NEQ> &a) {
                const bool past = t * PP + u >= len;
#pragma unroll
                for (int r = 0; r < NEQ; ++r) {
#pragma unroll
                    for (int c = 0; c < NEQ; ++c)
                        a.m[r + NEQ * c] = past ? (r == c ? (AT)1 : (AT)0) : C[u][r + NEQ * c];
                    a.v[r] = past ? (AT)0 : w[u][r];
                }
            },
            [&](int u, const AT *x) {
#pragma unroll
                for (int n = 0; n < NEQ; ++n) w[u][n] = x[n];
            },
            lb, lane, wv);
        if (AHEAD) load(C, pC, ln);
#pragma unroll
        for (int u = 0; u < PP; ++u) {
            const int v = t * PP + u;
#pragma unroll
            for (int n = 0; n < NEQ; ++n) {
                const double xd = (double)w[u][n];
                const double nv = assign ? xd : own[u][n] + underr * (xd - own[u][n]);
                if (v < len) dq[n * N + (long)l * len + v] = nv;
                done[u][n] = nv;
            }
        }
        lprev = l;
    }
}

// The walk of lines of up to NT points with three times the threads.  The matrices of a scan's
// steps, 27 of a step's 36 multiply-adds and 9 of its 12 exchanges, follow from the operands
// alone, so two more groups of waves, one for each direction, form them a line ahead and pass
// them through LDS, and the chain of lines is left with the vectors.  The forward matrices of line
// l + 1 are written between the barriers S1 and S2 of line l (one in each of its scans), the
// backward ones between S2 of line l and S1 of line l + 1, while the other direction's are read.
// FP32-LHS 945x241: an eta line (241 points) 2.4 us instead of 3.2, with one group for both
// directions 3.0.  The matrices of both directions take 432 bytes (FP64: 864) of LDS a point, so
// lines of up to 256 (128) points go this way, longer ones that of k_lr_walk.
template <typename T> struct ScanMats {   // one step's matrix of a lane, in 16-byte pieces
    static constexpr int W = 16 / sizeof(T), K = 9 / W;
    typedef T V __attribute__((ext_vector_type(W)));
};

template <typename LT, int NT> struct ScanLds {
    using S = ScanMats<LT>;
    typename S::V v[2][6][S::K][NT];   // direction, step (before step 1..5; after the last)
    LT x[2][6][NT];
};
template <typename LT, int NT>
SMAC_DEV void mats_put(ScanLds<LT, NT> &L, int dir, int step, int t, const LT *m)
{
    using S = ScanMats<LT>;
#pragma unroll
    for (int k = 0; k < S::K; ++k) {
        typename S::V p;
#pragma unroll
        for (int e = 0; e < S::W; ++e) p[e] = m[k * S::W + e];
        L.v[dir][step][k][t] = p;
    }
    L.x[dir][step][t] = m[8];
}
template <typename LT, int NT>
SMAC_DEV void mats_get(const ScanLds<LT, NT> &L, int dir, int step, int t, LT *m)
{
    using S = ScanMats<LT>;
#pragma unroll
    for (int k = 0; k < S::K; ++k) {
        const typename S::V p = L.v[dir][step][k][t];
#pragma unroll
        for (int e = 0; e < S::W; ++e) m[k * S::W + e] = p[e];
    }
    m[8] = L.x[dir][step][t];
}

// a step of the matrices; of the vectors, whose matrix of this lane is m
template <typename AT, bool FWD, int OFF>
SMAC_DEV void mats_level(AT *m, int lane)
{
    Aff<AT, 3> n, o;
#pragma unroll
    for (int e = 0; e < 9; ++e) {
        n.m[e] = m[e];
        o.m[e] = lane_shift<OFF, FWD>(m[e], lane);
    }
#pragma unroll
    for (int e = 0; e < 3; ++e) n.v[e] = o.v[e] = (AT)0;
    aff_after(n, o);
    const bool has = FWD ? lane >= OFF : lane + OFF < 64;
#pragma unroll
    for (int e = 0; e < 9; ++e) m[e] = has ? n.m[e] : m[e];
}
template <typename AT, bool FWD, int OFF>
SMAC_DEV void vec_level(const AT *m, AT *v, int lane)
{
    AT o[3], n[3];
#pragma unroll
    for (int e = 0; e < 3; ++e) o[e] = lane_shift<OFF, FWD>(v[e], lane);
    aff_apply<AT, 3>(m, v, o, n);
    const bool has = FWD ? lane >= OFF : lane + OFF < 64;
#pragma unroll
    for (int e = 0; e < 3; ++e) v[e] = has ? n[e] : v[e];
}

// line_scan of one point a thread with the steps' matrices from LDS: point map (m, v), x the
// value after it
template <typename AT, int NT, bool FWD>
SMAC_DEV void line_scan_ahead(const AT *m, const AT *v0, AT *x, const ScanLds<AT, NT> &L, AT (*tot)[12],
                              int t)
{
    constexpr int NW = NT / 64, D = FWD ? 0 : 1;
    const int lane = t & 63, wv = t >> 6;
    AT a[6][9], v[3];
#pragma unroll
    for (int k = 0; k < 6; ++k) mats_get(L, D, k, t, a[k]);
#pragma unroll
    for (int n = 0; n < 3; ++n) v[n] = v0[n];
    vec_level<AT, FWD, 1>(m, v, lane);
    vec_level<AT, FWD, 2>(a[0], v, lane);
    vec_level<AT, FWD, 4>(a[1], v, lane);
    vec_level<AT, FWD, 8>(a[2], v, lane);
    vec_level<AT, FWD, 16>(a[3], v, lane);
    vec_level<AT, FWD, 32>(a[4], v, lane);
    if (lane == (FWD ? 63 : 0)) {
#pragma unroll
        for (int e = 0; e < 9; ++e) tot[wv][e] = a[5][e];
#pragma unroll
        for (int n = 0; n < 3; ++n) tot[wv][9 + n] = v[n];
    }
    __syncthreads();
    AT Y[3], ye[3], cur[3];
    wave_entry<AT, 3, NW, FWD>(tot, wv, Y);
    aff_apply<AT, 3>(a[5], v, Y, ye);
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        const AT nb = lane_shift<1, FWD>(ye[n], lane);
        cur[n] = lane == (FWD ? 0 : 63) ? Y[n] : nb;
    }
    aff_apply<AT, 3>(m, v0, cur, x);
}

template <typename LT, int NT>
__global__ void __launch_bounds__(3 * NT)
k_lr_walk_ahead(int nline, int len, long N, int count, int first, int step, double underr,
                double *__restrict__ dq, const double *__restrict__ s, const LT *__restrict__ op)
{
    constexpr int NB = 9, NW = NT / 64;
    __shared__ ScanLds<LT, NT> L;
    __shared__ LT lf[NW][12], lb[NW][12];
    const bool up = step > 0;
    const int t = threadIdx.x & (NT - 1), lane = t & 63;
    const bool in = t < len;
    const LT *pB = op, *pM = op + NB * N, *pC = op + 2 * NB * N,
             *pNear = op + (up ? 3 : 4) * NB * N, *pFar = op + (up ? 4 : 3) * NB * N;
    auto line = [&](int idx) {
        const int l = (first + (idx < count ? idx : count - 1) * step) % nline;
        return l < 0 ? l + nline : l;
    };
    // past the line's end in-range addresses stand, whose values nothing uses
    const int at0 = in ? t : len - 1;
    auto load = [&](LT *x, const LT *pl, int l) {
#pragma unroll
        for (int e = 0; e < NB; ++e) x[e] = pl[e * N + (long)l * len + at0];
    };
    // a point's map: past the line the identity
    auto map = [&](LT *x) {
#pragma unroll
        for (int e = 0; e < NB; ++e) x[e] = in ? x[e] : e % 4 == 0 ? (LT)1 : (LT)0;
    };
    // a direction's matrices, formed in registers while that direction's of the line before are
    // in use, then written to LDS
    auto produce = [&](auto fwd) {
        constexpr bool FWD = decltype(fwd)::value;
        constexpr int D = FWD ? 0 : 1;
        const LT *pl = FWD ? pM : pC;
        LT m[NB], a[6][NB];
        auto form = [&](int next) {
            map(m);
            auto keep = [&](int k) {
#pragma unroll
                for (int e = 0; e < NB; ++e) a[k][e] = m[e];
            };
            mats_level<LT, FWD, 1>(m, lane);
            keep(0);
            mats_level<LT, FWD, 2>(m, lane);
            keep(1);
            mats_level<LT, FWD, 4>(m, lane);
            keep(2);
            mats_level<LT, FWD, 8>(m, lane);
            keep(3);
            mats_level<LT, FWD, 16>(m, lane);
            keep(4);
            mats_level<LT, FWD, 32>(m, lane);
            keep(5);
            load(m, pl, line(next));
        };
        auto put = [&]() {
#pragma unroll
            for (int k = 0; k < 6; ++k) mats_put(L, D, k, t, a[k]);
        };
        load(m, pl, line(0));
        form(1);
        if (FWD) put();
        __syncthreads();   // S0
        for (int idx = 0; idx < count; ++idx) {
            if (FWD) form(idx + 2);
            else put();
            __syncthreads();   // S1
            if (FWD) put();
            else form(idx + 2);
            __syncthreads();   // S2
        }
    };
    const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    if (group == 1) return produce(std::true_type{});
    if (group == 2) return produce(std::false_type{});
    __builtin_amdgcn_s_setprio(3);
    LT B[NB], M[NB], C[NB], near[NB], far[NB];
    double rhs[3], fx[3], own[3], done[3];
    auto loadv = [&](double *x, const double *pl, int l) {
#pragma unroll
        for (int n = 0; n < 3; ++n) x[n] = pl[n * N + (long)l * len + at0];
    };
    // what a line needs before its scans
    auto fetch = [&](int l) {
        const int beyond = up ? l + 1 : l - 1;
        load(B, pB, l);
        load(near, pNear, l);
        load(far, pFar, l);
        loadv(rhs, s, l);
        loadv(fx, dq, beyond >= 0 && beyond < nline ? beyond : l);
    };
    fetch(line(0));
    load(M, pM, line(0));
    load(C, pC, line(0));
    int lprev = -2;
    __syncthreads();   // S0
    for (int idx = 0; idx < count; ++idx) {
        const int l = line(idx), ln = line(idx + 1);
        const bool hm = l > 0, hp = l < nline - 1;
        const bool regm = lprev == l - 1, regp = lprev == l + 1;
        double r[3];
        LT bv[3], w[3], x[3];
#pragma unroll
        for (int n = 0; n < 3; ++n) r[n] = rhs[n];
        if (hm) {
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                double y[3];
#pragma unroll
                for (int n = 0; n < 3; ++n) y[n] = regm ? done[n] : fx[n];
                double b = (double)(up ? near : far)[m] * y[0];
#pragma unroll
                for (int n = 1; n < 3; ++n) b = b + (double)(up ? near : far)[m + 3 * n] * y[n];
                r[m] = r[m] - b;
            }
        }
        if (hp) {
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                double y[3];
#pragma unroll
                for (int n = 0; n < 3; ++n) y[n] = regp ? done[n] : fx[n];
                double b = (double)(up ? far : near)[m] * y[0];
#pragma unroll
                for (int n = 1; n < 3; ++n) b = b + (double)(up ? far : near)[m + 3 * n] * y[n];
                r[m] = r[m] - b;
            }
        }
        LT rr[3];
#pragma unroll
        for (int n = 0; n < 3; ++n) rr[n] = (LT)r[n];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            LT acc = B[m] * rr[0];
#pragma unroll
            for (int n = 1; n < 3; ++n) acc = acc + B[m + 3 * n] * rr[n];
            bv[m] = in ? acc : (LT)0;
        }
        loadv(own, dq, l);
        fetch(ln);
        map(M);
        line_scan_ahead<LT, NT, true>(M, bv, w, L, lf, t);    // S1
        load(M, pM, ln);
        map(C);
#pragma unroll
        for (int n = 0; n < 3; ++n) w[n] = in ? w[n] : (LT)0;
        line_scan_ahead<LT, NT, false>(C, w, x, L, lb, t);    // S2
        load(C, pC, ln);
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            const double nv = own[n] + underr * ((double)x[n] - own[n]);
            if (in) dq[n * N + (long)l * len + t] = nv;
            done[n] = nv;
        }
        lprev = l;
    }
}

// ------------------------------------------------------------------------------------------
// natural (j fastest) <-> eta-major (k fastest) transposition of the three planes of N of one
// array, or of two in one launch: at these sizes a launch costs as much as its traffic (945x241
// 5.5 us for 11 MB)

constexpr int TT = 32;

__global__ void __launch_bounds__(256)
k_transpose(const double *__restrict__ src0, double *__restrict__ dst0,
            const double *__restrict__ src1, double *__restrict__ dst1, int rows, int cols, long N)
{
    // src plane: rows x cols, cols fastest; dst plane: cols x rows, rows fastest
    __shared__ double tile[TT][TT + 1];
    const long base = (long)(blockIdx.z % 3) * N;
    const double *src = blockIdx.z < 3 ? src0 : src1;
    double *dst = blockIdx.z < 3 ? dst0 : dst1;
    const int c0 = blockIdx.x * TT, r0 = blockIdx.y * TT;
    for (int rr = threadIdx.y; rr < TT; rr += 8) {
        const int r = r0 + rr, c = c0 + threadIdx.x;
        if (r < rows && c < cols) tile[rr][threadIdx.x] = src[base + (long)r * cols + c];
    }
    __syncthreads();
    for (int cc = threadIdx.y; cc < TT; cc += 8) {
        const int c = c0 + cc, r = r0 + threadIdx.x;
        if (r < rows && c < cols) dst[base + (long)c * rows + r] = tile[threadIdx.x][cc];
    }
}

static void transpose(hipStream_t sm, int rows, int cols, long N, const double *src, double *dst,
                      const double *src1 = nullptr, double *dst1 = nullptr)
{
    dim3 g((cols + TT - 1) / TT, (rows + TT - 1) / TT, src1 ? 6 : 3);
    hipLaunchKernelGGL(k_transpose, g, dim3(TT, 8), 0, sm, src, dst, src1, dst1, rows, cols, N);
}

// wake-cut injection (bcimpds single-rank branch, ref/bc.f:571-591) with ds and rhs in the
// eta-major layout; q stays natural, and the natural rhs, which differs from the eta-major one in
// these points only, gets their values too.  Pairs outside the row are skipped.
__global__ void k_wake_eta(long N, int jm, int km, int neqs, int npair, int base,
                           const int *__restrict__ pairs, const double *__restrict__ sq,
                           double *__restrict__ ds, double *__restrict__ rhs,
                           double *__restrict__ rhs_nat)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npair) return;
    const long jt = pairs[2 * i] - base, jb = pairs[2 * i + 1] - base;
    if (jt < 0 || jt >= jm || jb < 0 || jb >= jm) return;
    const long t0 = jt * km, t1 = jt * km + 1, b1 = jb * km + 1;   // (jt,0), (jt,1), (jb,1)
    for (int n = 0; n < neqs; ++n) {
        double snew = 0.5 * (sq[n * N + jt + jm] + sq[n * N + jb + jm]);
        double dsnew = 0.5 * (ds[n * N + t1] + ds[n * N + b1]);
        ds[n * N + t0] = snew + dsnew - sq[n * N + jt];
        rhs[n * N + t0] = rhs_nat[n * N + jt] = ds[n * N + t0];
    }
}

__global__ void k_zero(double *__restrict__ a, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long)gridDim.x * blockDim.x)
        a[i] = 0.0;
}

// ------------------------------------------------------------------------------------------

// Threads and points per line: a line of up to 64 points stays within one wave, which has no
// waves to wait for or chain (47 points FP64: 6.4 us a transposed step against 7.8 in 256
// threads); pairs of points keep lines of up to 1024 at two waves per SIMD.
// twist: the operand planes hold the twisted factorisation (the reference-order walk always
// takes the plain one)
enum SweepForm { SWEEP_COLOUR, SWEEP_WALK, SWEEP_TRANSPOSED };

template <typename LT, int NEQ, SweepForm FORM>
static void sweep_launch(hipStream_t sm, int nline, int len, long N, int count, int first,
                         int step, double underr, int assign, double *dq, const double *s,
                         const LT *op, bool twist, const LrTStep &ts = {})
{
#define SWT(LAUNCH)                                                                             \
    do {                                                                                       \
        if (len <= 64) LAUNCH(64, 1);                                                          \
        else if (len <= 256) LAUNCH(256, 1);                                                   \
        else if (len <= 512) LAUNCH(512, 1);                                                   \
        else if (len <= 1024) LAUNCH(512, 2);                                                  \
        else LAUNCH(1024, 2);                                                                  \
    } while (0)
#define WALK(NT, PPV)                                                                           \
    hipLaunchKernelGGL((k_lr_walk<LT, NEQ, NT, PPV>), dim3(1), dim3(NT), 0, sm, nline, len, N,  \
                       count, first, step, underr, assign, dq, s, op)
#define AHEAD(NT)                                                                               \
    hipLaunchKernelGGL((k_lr_walk_ahead<LT, NT>), dim3(1), dim3(3 * NT), 0, sm, nline, len, N,  \
                       count, first, step, underr, dq, s, op)
#define COLOUR(NT, PPV, TW, TR)                                                                 \
    hipLaunchKernelGGL((k_lr_sweep<LT, NEQ, NT, PPV, TW, TR>), dim3(count), dim3(NT), 0, sm,    \
                       nline, len, N, count, first, step, underr, assign, dq, s, op, ts)
#define TWISTED(NT, PPV) COLOUR(NT, PPV, true, false)
#define PLAIN(NT, PPV) COLOUR(NT, PPV, false, false)
#define TRANSPOSED(NT, PPV) COLOUR(NT, PPV, false, true)
    if constexpr (FORM == SWEEP_WALK) {
        if constexpr (NEQ == 3) {
            constexpr int MOST = sizeof(LT) == 4 ? 256 : 128;
            if (len <= 64) AHEAD(64);
            else if (len <= MOST) AHEAD(MOST);
            else if (len <= 256) {
                if constexpr (MOST < 256) WALK(256, 1);
            } else if (len <= 512) WALK(512, 1);
            else if (len <= 1024) WALK(512, 2);
            else WALK(1024, 2);
        } else SWT(WALK);
    }
    else if constexpr (FORM == SWEEP_TRANSPOSED) SWT(TRANSPOSED);
    else if (twist) SWT(TWISTED);
    else SWT(PLAIN);
#undef TRANSPOSED
#undef PLAIN
#undef TWISTED
#undef COLOUR
#undef AHEAD
#undef WALK
#undef SWT
}

// one sweep of lines (reference order: odd sweeps ascending, even descending, as
// ref/lrelax.f:249-275; zebra: the lines of even index, then those of odd index)
template <typename LT, int NEQ>
static void sweep(hipStream_t sm, int nline, int len, long N, int nsweep, bool zebra, bool twist,
                  double underr, double *dq, const double *s, const LT *op)
{
    if (zebra) {
        sweep_launch<LT, NEQ, SWEEP_COLOUR>(sm, nline, len, N, (nline + 1) / 2, 0, 2, underr, 0, dq, s,
                                     op, twist);
        sweep_launch<LT, NEQ, SWEEP_COLOUR>(sm, nline, len, N, nline / 2, 1, 2, underr, 0, dq, s, op,
                                     twist);
        return;
    }
    const bool rev = (nsweep / 2) * 2 == nsweep;
    sweep_launch<LT, NEQ, SWEEP_WALK>(sm, nline, len, N, nline, rev ? nline - 1 : 0, rev ? -1 : 1,
                                underr, 0, dq, s, op, false);
}

long lr_scan_bytes(const Dims &d)
{
    // 45 operand planes (FP64 size) per direction + eta-major s and dq + the SA's 5 planes
    return (long)(2 * lr_planes<3>() + 6 + lr_planes<1>()) * d.N * 8 + 4 * 256;
}

template <typename LT>
void launch_lr_factor3(hipStream_t sm, const Dims &d, bool xi, bool eta, bool twist,
                       const LT *btc, const LT *bjm, const LT *bjp, const LT *bkm, const LT *bkp,
                       LT *opx, LT *ope)
{
    const int lpx = lines_per_group(d.km, twist), lpe = lines_per_group(d.jm, twist);
    const int nx = xi ? (d.km + lpx - 1) / lpx : 0, ne = eta ? (d.jm + lpe - 1) / lpe : 0;
    if (nx + ne > 0)
        hipLaunchKernelGGL((k_lr_factor<LT, 3>), dim3(nx + ne), dim3(twist ? 2 * FW : FW), 0, sm, d,
                           nx, lpx, lpe, twist ? 1 : 0, btc, bjm, bjp, bkm, bkp, opx, ope);
}

template <typename LT>
void launch_lrelax_scan(hipStream_t sm, const Dims &d, const DevParams &prm, int njsp, int nksp,
                        int nbcimp, bool zebra, const WakePairs &w, const double *q, double *dq,
                        double *s, const LT *btc, const LT *bjm, const LT *bjp, const LT *bkm,
                        const LT *bkp, const LrScan &ws, bool factor, int twist)
{
    const long N = d.N;
    LT *opx = (LT *)ws.opx, *ope = (LT *)ws.ope;
    // the twisted factorisation for the zebra passes (unless the caller says otherwise);
    // the plain one for the reference-order walk
    const bool tw = zebra && twist != 0;
    hipLaunchKernelGGL(k_zero, dim3(256), dim3(256), 0, sm, dq, 3 * N);
    // both directions' factorisations depend on the blocks only: one launch
    if (factor)
        launch_lr_factor3<LT>(sm, d, njsp > 0, nksp > 0, tw, btc, bjm, bjp, bkm, bkp, opx, ope);
    for (int nj = 1; nj <= njsp; ++nj) {
        sweep<LT, 3>(sm, d.km, d.jm, N, nj, zebra, tw, prm.underr, dq, s, opx);
        if ((nj / nbcimp) * nbcimp == nj) launch_wake(sm, d, 3, w, q, dq, s);
    }
    if (nksp > 0) {
        transpose(sm, d.km, d.jm, N, s, ws.s_t, dq, ws.dq_t);
        for (int nk = 1; nk <= nksp; ++nk) {
            sweep<LT, 3>(sm, d.jm, d.km, N, nk, zebra, tw, prm.underr, ws.dq_t, ws.s_t, ope);
            if ((nk / nbcimp) * nbcimp == nk && w.n > 0)
                hipLaunchKernelGGL(k_wake_eta, dim3((w.n + 63) / 64), dim3(64), 0, sm, N, d.jm,
                                   d.km, 3, w.n, w.base, w.pairs, q, ws.dq_t, ws.s_t, s);
        }
        transpose(sm, d.jm, d.km, N, ws.dq_t, dq);
    }
}

// ------------------------------------------------------------------------------------------
// the transpose of the zebra sweeps (the adjoint's preconditioner).  The sweeps map the
// right-hand side s to dq linearly (dq starts at zero; one colour step replaces dq_l on the
// lines of its colour by (1-w) dq_l + w T_l^-1 (s_l - Om_l dq_(l-1) - Op_l dq_(l+1))).  Their
// transpose runs the colour steps in reverse order, each transposed: with a the adjoint of
// dq and z_l = T_l^-T a_l on the colour's lines (a plain line solve of the transposed line
// system, whose factorisation is that of the transposed and shifted blocks),
//     sbar_l += w z_l,   a_l <- (1-w) a_l                 (lines of the colour)
//     a_m -= w (Om'_m z_(m-1) + Op'_m z_(m+1))            (the other lines)
// where Om'_m = (Op_(m-1))^T and Op'_m = (Om_(m+1))^T are again the transposed system's
// blocks to the neighbouring lines at the point.

//
// A step's line solves are one launch: a line first takes the terms of the z that the step
// before left on its neighbours (LrTStep::spread), is solved, and adds to its sbar and scales
// its a from what the workgroup holds.  The terms that the last step leaves to the other
// colour are taken on the way back to the natural layout (k_lr_tback).  A pair of kernels per
// step, solve and spread, took 7.7 + 4.9 us at 203x47; a xi step takes 8.3, an eta step 6.4.

// after the last eta step: out = sbar and, with planes 3..5, a = at less the terms of z on the
// lines of odd index, eta-major to natural
template <typename LT>
__global__ void __launch_bounds__(256)
k_lr_tback(int nline, int len, long N, double w, const double *__restrict__ at,
           const double *__restrict__ sbar, const double *__restrict__ z,
           const LT *__restrict__ op, double *__restrict__ a, double *__restrict__ out)
{
    __shared__ double tile[TT][TT + 1];
    const LT *pOm = op + 27 * N, *pOp = op + 36 * N;
    const int m = blockIdx.z % 3;
    const bool second = blockIdx.z >= 3;
    const int c0 = blockIdx.x * TT, r0 = blockIdx.y * TT;
    for (int rr = threadIdx.y; rr < TT; rr += 8) {
        const int l = r0 + rr, c = c0 + threadIdx.x;
        if (l >= nline || c >= len) continue;
        const long o = (long)l * len + c;
        double v = (second ? at : sbar)[m * N + o];
        if (second && (l & 1)) {
            double acc = 0.0;
#pragma unroll
            for (int k = 0; k < 3; ++k) acc += (double)pOm[(m + 3 * k) * N + o] * z[k * N + o - len];
            if (l < nline - 1) {
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    acc += (double)pOp[(m + 3 * k) * N + o] * z[k * N + o + len];
            }
            v -= w * acc;
        }
        tile[rr][threadIdx.x] = v;
    }
    __syncthreads();
    for (int cc = threadIdx.y; cc < TT; cc += 8) {
        const int c = c0 + cc, l = r0 + threadIdx.x;
        if (l < nline && c < len)
            (second ? a : out)[m * N + (long)c * nline + l] = tile[threadIdx.x][cc];
    }
}

// begin: sbar starts from zero with each colour's first step
template <typename LT>
static void tsweep(hipStream_t sm, int nline, int len, long N, int nsweep, double w, double *a,
                   double *sbar, double *z, const LT *op, bool begin)
{
    for (int sw = 0; sw < nsweep; ++sw)
        for (int par = 1; par >= 0; --par) {
            const LrTStep ts{a, sbar, w, sw > 0 || par == 0, begin && sw == 0};
            const int count = par ? nline / 2 : (nline + 1) / 2;
            if (count > 0)
                sweep_launch<LT, 3, SWEEP_TRANSPOSED>(sm, nline, len, N, count, par, 2, 1.0, 1, z,
                                                      nullptr, op, false, ts);
        }
}

template <typename LT>
void launch_lrelax_scan_t(hipStream_t sm, const Dims &d, int njsp, int nksp, double underr,
                          double *out, const LrScan &wt, const LrTWork &v)
{
    const long N = d.N;
    // the eta sweeps came last in the primal: their transposes come first
    if (nksp > 0) {
        const LT *op = (const LT *)wt.ope;
        tsweep<LT>(sm, d.jm, d.km, N, nksp, underr, v.at, v.st, v.zt, op, true);
        const dim3 g((d.km + TT - 1) / TT, (d.jm + TT - 1) / TT, njsp > 0 ? 6 : 3);
        hipLaunchKernelGGL(k_lr_tback<LT>, g, dim3(TT, 8), 0, sm, d.jm, d.km, N, underr, v.at,
                           v.st, v.zt, op, v.a, out);
    } else if (njsp == 0) {
        hipLaunchKernelGGL(k_zero, dim3(256), dim3(256), 0, sm, out, 3 * N);
    }
    if (njsp > 0)
        tsweep<LT>(sm, d.km, d.jm, N, njsp, underr, v.a, out, v.z, (const LT *)wt.opx, nksp == 0);
}

void launch_sa_lreltur_scan(hipStream_t sm, const Dims &d, int ntjsp, const WakePairs &w,
                            SaArrays &a, const LrScan &ws)
{
    // lreltur (ref/lreltur.f:52-252): ds = 0; ntjsp passes of the k lines in ascending order
    // followed by a re-solve of line k = 1, each pass ending with the wake injection.  With
    // the zebra order (that of the mean flow) a pass takes the even lines, the odd lines, and
    // then line k = 1 again.
    hipLaunchKernelGGL(k_zero, dim3(256), dim3(256), 0, sm, a.ds, d.N);
    const int lpx = lines_per_group(d.km, ws.zebra), nx = (d.km + lpx - 1) / lpx;
    hipLaunchKernelGGL((k_lr_factor<double, 1>), dim3(nx), dim3(ws.zebra ? 2 * FW : FW), 0, sm, d, nx,
                       lpx, lpx, ws.zebra ? 1 : 0, a.stc, a.sjm, a.sjp, a.skm, a.skp, ws.sa_op,
                       (double *)nullptr);
    for (int pass = 1; pass <= ntjsp; ++pass) {
        if (ws.zebra) {
            sweep_launch<double, 1, SWEEP_COLOUR>(sm, d.km, d.jm, d.N, (d.km + 1) / 2, 0, 2, 1.0, 1,
                                           a.ds, a.sf, ws.sa_op, true);
            sweep_launch<double, 1, SWEEP_COLOUR>(sm, d.km, d.jm, d.N, d.km / 2, 1, 2, 1.0, 1, a.ds,
                                           a.sf, ws.sa_op, true);
            sweep_launch<double, 1, SWEEP_COLOUR>(sm, d.km, d.jm, d.N, 1, 0, 1, 1.0, 1, a.ds, a.sf,
                                           ws.sa_op, true);
        } else {
            sweep_launch<double, 1, SWEEP_WALK>(sm, d.km, d.jm, d.N, d.km + 1, 0, 1, 1.0, 1, a.ds, a.sf,
                                          ws.sa_op, false);
        }
        launch_wake(sm, d, 1, w, a.anut, a.ds, a.sf);
    }
}

template void launch_lr_factor3<double>(hipStream_t, const Dims &, bool, bool, bool, const double *,
                                        const double *, const double *, const double *,
                                        const double *, double *, double *);
template void launch_lrelax_scan_t<double>(hipStream_t, const Dims &, int, int, double, double *,
                                           const LrScan &, const LrTWork &);
template void launch_lrelax_scan<double>(hipStream_t, const Dims &, const DevParams &, int, int,
                                         int, bool, const WakePairs &, const double *, double *,
                                         double *, const double *, const double *,
                                         const double *, const double *, const double *,
                                         const LrScan &, bool, int);
template void launch_lrelax_scan<float>(hipStream_t, const Dims &, const DevParams &, int, int,
                                        int, bool, const WakePairs &, const double *, double *,
                                        double *, const float *, const float *, const float *,
                                        const float *, const float *, const LrScan &, bool, int);

}  // namespace smac
