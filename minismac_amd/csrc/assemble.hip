// Residual and implicit-operator assembly of one pass of the implicit iteration:
// conup + fluxj3/fluxk3 (ref/conup.f:49-478, ref/flux.f:160-372), viscterms
// (ref/visc.f:50-160), boundary blanking and the pseudo-time diagonal (ref/step.f:386-437),
// the BC rows of bcmain (ref/bc.f:60-224 and the routines it calls), and resid + rhsnorm
// (ref/step.f:613-756, 513-519).
//
// A point needs the flux-split face Jacobians A+/A- of its four xi faces and four eta faces
// (the third-order flux of a face reads dfp/dfm of the faces either side), the point Jacobians
// of its neighbours and the constant-viscosity face coefficients, and writes s (3 planes) and
// the five 3x3 blocks (45 planes) once: 448 bytes a point in FP64, which the memory takes in
// 21 us at 945x241 and 83 at 1889x481.  A face is 230 FP64 instructions with five divisions and
// a root.  With every point computing its eight faces the kernel was bound by those (41 and
// 197 us, FP32-LHS batch of 1.2 M points 242); b_assemble below computes each face about once
// (30, 117 and 169).
#include "smac_dev.h"
#include "smac_kernels.h"

#include <type_traits>

namespace smac {

// ---------------------------------------------------------------------------------------
// face split, ref/conup.f:127-185 (xi) and :306-355 (eta); rt (time metric) is zero for the
// static grids of this path (ref/metric.f:244-248), kept in the expressions as 0.0
struct Face {
    double ap[9], am[9];   // (m + 3n)
};

SMAC_DEV void face_split(double rx, double ry, double q2, double q3, double beta, Face &f)
{
    const double rt = 0.0;
    double cvel = rx * q2 + ry * q3;
    double t = cvel + 0.5 * rt;
    double cc = sqrt(t * t + beta * (rx * rx + ry * ry));
    double eig = cvel + rt;
    double eig1 = 0.5 * (eig + fabs(eig));
    double eig2 = cvel + rt * 0.5 + cc;
    double x21 = -ry * eig1 / (cc * cc - 0.25 * rt * rt);
    double x31 = rx * eig1 / (cc * cc - 0.25 * rt * rt);
    double x12 = 0.5 * eig2 / cc;
    double x22 = 0.5 * eig2 * (q2 * eig2 + beta * rx) / (beta * cc * (cc - 0.5 * rt));
    double x32 = 0.5 * eig2 * (q3 * eig2 + beta * ry) / (beta * cc * (cc - 0.5 * rt));
    double xi11 = ry * q2 - rx * q3;
    double xi12 = -q3 * (cvel + rt) - ry * beta;
    double xi13 = q2 * (cvel + rt) + rx * beta;
    double xi21 = cc - cvel - 0.5 * rt;
    double xi22 = rx * beta;
    double xi23 = ry * beta;
    f.ap[0] = x12 * xi21;
    f.ap[1] = x21 * xi11 + x22 * xi21;
    f.ap[2] = x31 * xi11 + x32 * xi21;
    f.ap[3] = x12 * xi22;
    f.ap[4] = x21 * xi12 + x22 * xi22;
    f.ap[5] = x31 * xi12 + x32 * xi22;
    f.ap[6] = x12 * xi23;
    f.ap[7] = x21 * xi13 + x22 * xi23;
    f.ap[8] = x31 * xi13 + x32 * xi23;
    f.am[0] = -f.ap[0];
    f.am[1] = -f.ap[1] + rx;
    f.am[2] = -f.ap[2] + ry;
    f.am[3] = -f.ap[3] + rx * beta;
    f.am[4] = -f.ap[4] + rt + 2. * rx * q2 + ry * q3;
    f.am[5] = -f.ap[5] + rx * q3;
    f.am[6] = -f.ap[6] + ry * beta;
    f.am[7] = -f.ap[7] + ry * q2;
    f.am[8] = -f.ap[8] + rt + rx * q2 + 2. * ry * q3;
}

// point flux Jacobian, ref/conup.f:89-105
SMAC_DEV void point_jac(double rx, double ry, double u, double v, double beta, double at[9])
{
    const double rt = 0.0;
    double cvel = rt + rx * u + ry * v;
    at[0] = rt;
    at[1] = rx;
    at[2] = ry;
    at[3] = rx * beta;
    at[4] = rx * u + cvel;
    at[5] = rx * v;
    at[6] = ry * beta;
    at[7] = ry * u;
    at[8] = ry * v + cvel;
}

// physical flux of a point, ref/flux.f:177-181
SMAC_DEV void point_flux(double p, double u, double v, double rx, double ry, double beta,
                         double fv[3])
{
    const double rt = 0.0;
    double cvel = rt + rx * u + ry * v;
    fv[0] = rt * p + beta * (cvel - rt);
    fv[1] = u * cvel + rx * p;
    fv[2] = v * cvel + ry * p;
}

// what a point's stencil needs of it
struct Pt {
    double p, u, v, dj, xix, xiy, etx, ety;
};

// element j of the row at `row`, the same for all lanes: a 32-bit byte offset to a scalar base
template <typename T> SMAC_DEV T &at_lane(T *row, unsigned j)
{
    using C = typename std::conditional<std::is_const<T>::value, const char, char>::type;
    return *(T *)((C *)row + j * (unsigned)sizeof(T));
}

// point j of the row that starts at point o
SMAC_DEV void load_pt(const double *__restrict__ q, const double *__restrict__ met,
                      const double *__restrict__ dj, long N, long o, unsigned j, Pt &t)
{
    t.p = at_lane(q + o, j);
    t.u = at_lane(q + o + N, j);
    t.v = at_lane(q + o + 2 * N, j);
    t.dj = at_lane(dj + o, j);
    t.xix = at_lane(met + o, j);
    t.xiy = at_lane(met + o + N, j);
    t.etx = at_lane(met + o + 2 * N, j);
    t.ety = at_lane(met + o + 3 * N, j);
}

// one face of one direction, between points a and b (a first): the split Jacobians, the
// differences they take (d: dfp, then dfm), and the viscous coefficients, default REAL
// (ref/visc.f:95-113)
struct FaceVals {
    Face F;
    double d[6];
};
SMAC_DEV void face_vals(const Pt &a, const Pt &b, double rxa, double rya, double rxb, double ryb,
                        double beta, FaceVals &f)
{
    const double rx = 0.5 * (rxb + rxa);
    const double ry = 0.5 * (ryb + rya);
    const double q2 = 0.5 * (b.u + a.u);
    const double q3 = 0.5 * (b.v + a.v);
    face_split(rx, ry, q2, q3, beta, f.F);
    const double dq1 = b.p - a.p;
    const double dq2 = b.u - a.u;
    const double dq3 = b.v - a.v;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        f.d[m] = f.F.ap[m] * dq1 + f.F.ap[m + 3] * dq2 + f.F.ap[m + 6] * dq3;
        f.d[3 + m] = f.F.am[m] * dq1 + f.F.am[m + 3] * dq2 + f.F.am[m + 6] * dq3;
    }
}
struct Visc {
    float vf, ud, vd;
};
SMAC_DEV Visc face_visc(const Pt &a, const Pt &b, double rxa, double rya, double rxb, double ryb,
                        double vnu)
{
    const double djv = 0.5 * (a.dj * vnu + b.dj * vnu);
    const double rx = 0.5 * (rxa + rxb);
    const double ry = 0.5 * (rya + ryb);
    return Visc{(float)(djv * (rx * rx + ry * ry)), (float)(b.u - a.u), (float)(b.v - a.v)};
}

// the numerical flux of face f of a line of n points (flux.f): fv0, fv1 the physical fluxes of
// its two points, dm, dc, dp the differences of faces f-1, f and f+1.  The reference clamps
// the neighbour faces' indices; the coefficients cp, cm vanish where it does (face 0's own
// differences stand for face -1's, zeros for those of the face past the last).
SMAC_DEV void face_flux(int f, int n, double cdis, const double fv0[3], const double fv1[3],
                        const double dm[6], const double dc[6], const double dp[6], double ff[3])
{
    const double r6 = (double)(1.0f / 6.0f);   // a default-REAL quotient in the reference
    const int fm = f - 1 > 0 ? f - 1 : 0;
    const int fp = f + 1 < n - 1 ? f + 1 : n - 1;
    const int fpp = f + 2 < n - 1 ? f + 2 : n - 1;
    const float cp = (float)(fpp - fp);
    const float cm = (float)(f - fm);
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const double pc = dc[m], mc = dc[3 + m];
        const double pn = dp[m], mn = dp[3 + m];
        const double pm = f == 0 ? pc : dm[m], mm = f == 0 ? mc : dm[3 + m];
        const double fmn = (pc + mc - pn - mn) * r6;
        const double fpl = (pm + mm - pc - mc) * r6;
        const double f3 = (pm - pc + mc - mn) * r6;
        ff[m] = 0.5 * (fv1[m] + fv0[m]) +
                cdis * ((double)(cp * cm) * f3 + (double)(cm * (1.f - cp)) * fpl +
                        (double)(cp * (1.f - cm)) * fmn);
    }
}

// a neighbouring lane's value: lane-1 (wave_shr) or lane+1 (wave_shl)
template <bool UP> SMAC_DEV int from_lane(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, UP ? 0x138 : 0x130, 0xf, 0xf, true);
}
template <bool UP> SMAC_DEV float from_lane(float v)
{
    return __builtin_bit_cast(float, from_lane<UP>(__builtin_bit_cast(int, v)));
}
template <bool UP> SMAC_DEV double from_lane(double v)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)from_lane<UP>((int)(unsigned)u);
    const unsigned hi = (unsigned)from_lane<UP>((int)(unsigned)(u >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

constexpr int ASM_COLS = 60;   // points of a row that a wave assembles

// One wave assembles ASM_COLS points of `rows` rows, lane l at j = ASM_COLS bk.x + l - 2, and
// marches in k.  A lane computes the xi face between its point and the next and one eta face
// per row; what a point needs of its other faces comes from the lanes beside it (DPP moves; the
// two outer lanes on each side only serve their neighbours) and from the rows
// before (registers).  The row r's blocks need the eta faces r-1 and r; s of row r-1 needs the
// fluxes of faces r-2 and r-1, which need face r: so s follows its blocks by one row, and a
// strip starts two faces early and ends one late.
template <typename LT>
SMAC_DEV void b_assemble(const Blk &bk, int rows, const Dims &d, const DevParams &prm,
                         const double *__restrict__ q, const double *__restrict__ met,
                         const double *__restrict__ dj, double *__restrict__ s,
                         LT *__restrict__ btc, LT *__restrict__ bjm, LT *__restrict__ bjp,
                         LT *__restrict__ bkm, LT *__restrict__ bkp)
{
    const int lane = threadIdx.x & 63, jm = d.jm, km = d.km;
    const int j = ASM_COLS * (int)bk.x + lane - 2;
    const int r0 = rows * (int)bk.y, r1 = r0 + rows < km ? r0 + rows : km;   // rows [r0, r1)
    const long N = d.N;
    const int jc = j < 0 ? 0 : (j > jm - 1 ? jm - 1 : j);
    const bool out = lane >= 2 && lane < 2 + ASM_COLS && j < jm;
    const bool jin = j > 0 && j < jm - 1, jface = j >= 0 && j < jm - 1;
    const double beta = prm.beta;
    auto fetch = [&](int r, Pt &t) {
        const int rc = r < 0 ? 0 : (r > km - 1 ? km - 1 : r);
        load_pt(q, met, dj, N, (long)rc * jm, (unsigned)jc, t);
    };
    Pt cur, nxt, pre;        // rows r, r+1, r+2
    fetch(r0 - 2, cur);
    fetch(r0 - 1, nxt);
    // of the faces and rows before: differences of faces r-2 and r-1, split of face r-1, flux
    // of face r-2, physical flux of point r, point r-1's Jacobian operands, viscous faces r-2
    // and r-1, and of row r-1 the xi terms of s
    double d2[6] = {}, d1[6] = {}, ap0[9] = {}, am0[9] = {}, ff2[3] = {}, fv0[3] = {};
    double pu = 0.0, pv = 0.0, prx = 0.0, pry = 0.0, sx[3] = {};
    Visc v2{0.f, 0.f, 0.f}, v1{0.f, 0.f, 0.f};
    float tx2 = 0.f, tx3 = 0.f;
    for (int r = r0 - 2; r <= r1; ++r) {
        fetch(r + 2, pre);
        const bool mine = r >= r0 && r < r1, inner = r > 0 && r < km - 1;
        // the planes' addresses are formed anew in each row (two scalar additions each): kept
        // over the loop, 48 of them do not fit the scalar registers
        long N = d.N;
        asm volatile("" : "+s"(N));
        const long o = (long)r * jm;
        double vc[9], sxn[3];
        Visc vr{0.f, 0.f, 0.f}, vl{0.f, 0.f, 0.f};
        if (mine && inner) {
            // ---- xi: the face to the next point, then what the lane before holds
            // (ref/conup.f:216-271, ref/visc.f:95-113)
            Pt right;
            right.p = from_lane<false>(cur.p);
            right.u = from_lane<false>(cur.u);
            right.v = from_lane<false>(cur.v);
            right.dj = from_lane<false>(cur.dj);
            right.xix = from_lane<false>(cur.xix);
            right.xiy = from_lane<false>(cur.xiy);
            FaceVals x;
            face_vals(cur, right, cur.xix, cur.xiy, right.xix, right.xiy, beta, x);
#pragma unroll
            for (int i = 0; i < 6; ++i) x.d[i] = jface ? x.d[i] : 0.0;
            {
                double dl[6], dr[6], fc[3], fr[3], fx[3];
#pragma unroll
                for (int i = 0; i < 6; ++i) {
                    dl[i] = from_lane<true>(x.d[i]);
                    dr[i] = from_lane<false>(x.d[i]);
                }
                point_flux(cur.p, cur.u, cur.v, cur.xix, cur.xiy, beta, fc);
#pragma unroll
                for (int m = 0; m < 3; ++m) fr[m] = from_lane<false>(fc[m]);
                face_flux(j, jm, prm.cdis, fc, fr, dl, x.d, dr, fx);
#pragma unroll
                for (int m = 0; m < 3; ++m) sxn[m] = -(fx[m] - from_lane<true>(fx[m]));
            }
            double a4 = 0.0, b4 = 0.0;
            if (prm.ivis == 1) {
                vr = face_visc(cur, right, cur.xix, cur.xiy, right.xix, right.xiy, prm.vnu);
                vl.vf = from_lane<true>(vr.vf);
                vl.ud = from_lane<true>(vr.ud);
                vl.vd = from_lane<true>(vr.vd);
                a4 = vl.vf;
                b4 = vr.vf;
            }
            double al[9], ar[9];
            point_jac(from_lane<true>(cur.xix), from_lane<true>(cur.xiy), from_lane<true>(cur.u),
                      from_lane<true>(cur.v), beta, al);
            point_jac(right.xix, right.xiy, right.u, right.v, beta, ar);
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                const double apl = from_lane<true>(x.F.ap[i]), aml = from_lane<true>(x.F.am[i]);
                double bm = 0.5 * (-al[i] - apl + aml);
                double bp = 0.5 * (ar[i] - x.F.ap[i] + x.F.am[i]);
                vc[i] = 0.5 * (x.F.ap[i] + apl - x.F.am[i] - aml);
                if ((i == 4 || i == 8) && prm.ivis == 1) {
                    bm = bm - a4;
                    bp = bp - b4;
                }
                if (jin && out) {
                    at_lane(bjm + i * N + o, (unsigned)j) = (LT)bm;
                    at_lane(bjp + i * N + o, (unsigned)j) = (LT)bp;
                }
            }
        }
        // the eta face r, where it exists; elsewhere the reference reads it only as 0*stale
        FaceVals e;
        Visc ve{0.f, 0.f, 0.f};
        if (r >= 0 && r < km - 1) {
            face_vals(cur, nxt, cur.etx, cur.ety, nxt.etx, nxt.ety, beta, e);
            if (prm.ivis == 1) ve = face_visc(cur, nxt, cur.etx, cur.ety, nxt.etx, nxt.ety, prm.vnu);
        } else {
#pragma unroll
            for (int i = 0; i < 6; ++i) e.d[i] = 0.0;
#pragma unroll
            for (int i = 0; i < 9; ++i) e.F.ap[i] = e.F.am[i] = 0.0;
        }
        double fv1[3];
        point_flux(cur.p, cur.u, cur.v, cur.etx, cur.ety, beta, fv1);
        // flux of face r-1, between points r-1 and r
        double ff[3] = {0.0, 0.0, 0.0};
        if (r >= r0 && r > 0) face_flux(r - 1, km, prm.cdis, fv0, fv1, d2, d1, e.d, ff);
        // s of row r-1 (ref/conup.f:216-271, 377-457, ref/visc.f:95-140)
        if (r > r0) {
            double vs[3];
#pragma unroll
            for (int m = 0; m < 3; ++m) vs[m] = sx[m] - (ff[m] - ff2[m]);
            if (prm.ivis == 1) {
                vs[1] = vs[1] + (double)tx2;
                vs[2] = vs[2] + (double)tx3;
                const float t2 = v1.vf * v1.ud - v2.vf * v2.ud;
                const float t3 = v1.vf * v1.vd - v2.vf * v2.vd;
                vs[1] = vs[1] + (double)t2;
                vs[2] = vs[2] + (double)t3;
            }
            const bool live = jin && r - 1 > 0 && r - 1 < km - 1;
            if (out) {
#pragma unroll
                for (int m = 0; m < 3; ++m)
                    at_lane(s + m * N + o - jm, (unsigned)j) = live ? vs[m] : 0.0;
            }
        }
        if (mine && inner) {
            // ---- eta: add (ref/conup.f:377-457, ref/visc.f:121-140)
            double am_[9], ar[9];
            point_jac(prx, pry, pu, pv, beta, am_);
            point_jac(nxt.etx, nxt.ety, nxt.u, nxt.v, beta, ar);
            // pseudo-time diagonal (ref/step.f:419-437), fib = 1
            const double rdjdtau = 1.0 / (cur.dj * prm.dtau) + 1. - 1.0;
            const double xa = vl.vf, xb = vr.vf, a = v1.vf, b = ve.vf;
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                double bm = 0.5 * (-am_[i] - ap0[i] + am0[i]);
                double bp = 0.5 * (ar[i] - e.F.ap[i] + e.F.am[i]);
                double c = vc[i] + 0.5 * (e.F.ap[i] + ap0[i] - e.F.am[i] - am0[i]);
                if ((i == 4 || i == 8) && prm.ivis == 1) {
                    bm = bm - a;
                    bp = bp - b;
                    c = c + xa + xb;
                    c = c + a + b;
                }
                if (i == 0 || i == 4 || i == 8) c = c + rdjdtau;
                if (jin && out) {
                    at_lane(bkm + i * N + o, (unsigned)j) = (LT)bm;
                    at_lane(bkp + i * N + o, (unsigned)j) = (LT)bp;
                    at_lane(btc + i * N + o, (unsigned)j) = (LT)c;
                }
            }
#pragma unroll
            for (int m = 0; m < 3; ++m) sx[m] = sxn[m];
            tx2 = vr.vf * vr.ud - vl.vf * vl.ud;
            tx3 = vr.vf * vr.vd - vl.vf * vl.vd;
        }
        if (mine && out && !(jin && inner)) {
            // blanked boundary row: all blocks zero, btc = identity (ref/step.f:386-437)
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                at_lane(btc + i * N + o, (unsigned)j) = (LT)((i == 0 || i == 4 || i == 8) ? 1.0 : 0.0);
                at_lane(bjm + i * N + o, (unsigned)j) = (LT)0.0;
                at_lane(bjp + i * N + o, (unsigned)j) = (LT)0.0;
                at_lane(bkm + i * N + o, (unsigned)j) = (LT)0.0;
                at_lane(bkp + i * N + o, (unsigned)j) = (LT)0.0;
            }
        }
        // one row on
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            d2[i] = d1[i];
            d1[i] = e.d[i];
        }
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            ap0[i] = e.F.ap[i];
            am0[i] = e.F.am[i];
        }
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            ff2[m] = ff[m];
            fv0[m] = fv1[m];
        }
        v2 = v1;
        v1 = ve;
        pu = cur.u; pv = cur.v; prx = cur.etx; pry = cur.ety;
        cur = nxt;
        nxt = pre;
    }
}

// Rows per wave: marching saves faces (five a point for one row, 2.8 for four), one row each keeps
// more waves running; four rows where that still leaves the chip's 1024 SIMDs a wave each, two
// or one below.  1, 2, 4, 8 rows: 477x121 14.4, 19, 24, 40 us; 945x241 36, 30, 36, 50;
// 1889x481 188, 154, 117, 149.  A wave's 300 registers leave room for one per SIMD; held to
// two (256, a few spilled) it is the slower alone (120 us) and the faster in a batch (169 us
// against 190), whose blocks are unequal.
static int asm_rows(const Dims &d)
{
    const long strips = (d.jm + ASM_COLS - 1) / ASM_COLS;
    for (int rows = 4; rows > 1; rows /= 2)
        if (strips * ((d.km + rows - 1) / rows) >= 1024) return rows;
    return 1;
}

template <typename LT>
__global__ void __launch_bounds__(64)
k_assemble(Dims d, DevParams prm, int rows, const double *__restrict__ q,
           const double *__restrict__ met, const double *__restrict__ dj, double *__restrict__ s, LT *__restrict__ btc,
           LT *__restrict__ bjm, LT *__restrict__ bjp, LT *__restrict__ bkm, LT *__restrict__ bkp)
{
    b_assemble<LT>(xcd_blk(), rows, d, prm, q, met, dj, s, btc, bjm, bjp, bkm, bkp);
}

// ---------------------------------------------------------------------------------------
// BC rows (ref/bc.f): BC_MAX regions of the case in one launch, more in further ones in file
// order (in a batch too).  A region writes only its own points' rows and reads nothing that a
// region writes, so regions meet only in the points they share: one thread does all of a point's
// regions in the launch, in file order, and a later region's rows win as in the reference's
// sequence of calls.
//
// Bound by the latency of one point's chain of loads and of the far field's cosine, sine and
// divisions: 4.8 us at 945x241 and 10.5 at 1889x481 beside the SA,
// where one workgroup walking the regions, a barrier after each, took 15.5 and 42.

// bcoutj, extrapolation branch of ibval 31 plus the fixed-pressure row (ref/bc.f:1627-1676)
template <typename LT>
SMAC_DEV void bc_outj(const Dims &d, int j, int k, double pout, const double *__restrict__ q,
                      double *__restrict__ s, LT *btc, LT *bjm, LT *bjp)
{
    const long N = d.N, p = P(d, j, k);
    const int jn = j == 0 ? j + 1 : j - 1;
    LT *bn = j == 0 ? bjp : bjm;
    const long pn = P(d, jn, k);
    btc[4 * N + p] = (LT)1.0;
    btc[8 * N + p] = (LT)1.0;
    bn[4 * N + p] = (LT)-1.0;
    bn[8 * N + p] = (LT)-1.0;
    s[N + p] = q[N + pn] - q[N + p];
    s[2 * N + p] = q[2 * N + pn] - q[2 * N + p];
    btc[p] = (LT)1.0;
    s[p] = pout - q[p];
}

// bcnoslk, ibval 0 branch (ref/bc.f:1147-1158)
template <typename LT>
SMAC_DEV void bc_noslk(const Dims &d, int j, int k, const double *__restrict__ q,
                       double *__restrict__ s, LT *btc, LT *bkp)
{
    const long N = d.N, p = P(d, j, k), pu = P(d, j, k + 1);
    btc[p] = (LT)1.0;
    btc[4 * N + p] = (LT)1.0;
    btc[8 * N + p] = (LT)1.0;
    bkp[p] = (LT)-1.0;
    s[p] = q[pu] - q[p];
    s[N + p] = -q[N + p];
    s[2 * N + p] = -q[2 * N + p];
}

// bccgridk, ibval 25 at k = kmax: free stream plus a point vortex of strength clift for
// u, v and the outgoing characteristic for p (ref/bc.f:1334-1431)
template <typename LT>
SMAC_DEV void bc_cgridk(const Dims &d, int j, int k, double alpha, double beta, double clift,
                        const double *__restrict__ x, const double *__restrict__ y,
                        const double *__restrict__ met, const double *__restrict__ q,
                        double *__restrict__ s, LT *btc, LT *bkm)
{
    const long N = d.N, p = P(d, j, k), pd = P(d, j, k - 1);
    double pi = 4.0 * atan(1.0);
    double uinf = cos(alpha * pi / 180.);
    double vinf = sin(alpha * pi / 180.);
    double dx = x[p] - 0.25;
    double dy = y[p];
    double ucirc = clift * dy / (4. * pi * (dx * dx + dy * dy));
    double vcirc = -clift * dx / (4. * pi * (dx * dx + dy * dy));
    btc[4 * N + p] = (LT)1.0;
    btc[8 * N + p] = (LT)1.0;
    s[N + p] = uinf + ucirc - q[N + p];
    s[2 * N + p] = vinf + vcirc - q[2 * N + p];
    double r2 = met[2 * N + p], r3 = met[3 * N + p];
    double qq = r2 * q[N + p] + r3 * q[2 * N + p];
    double cc = sqrt(qq * qq + beta * (r2 * r2 + r3 * r3));
    double b11 = -(r2 * r2 + r3 * r3);
    double b12 = -r2 * (qq + cc);
    double b13 = -r3 * (qq + cc);
    bkm[p] = (LT)b11;
    bkm[3 * N + p] = (LT)b12;
    bkm[6 * N + p] = (LT)b13;
    btc[p] = (LT)(-b11);
    btc[3 * N + p] = (LT)(-b12);
    btc[6 * N + p] = (LT)(-b13);
    double dq1 = q[p] - q[pd];
    double dq2 = q[N + p] - q[N + pd];
    double dq3 = q[2 * N + p] - q[2 * N + pd];
    s[p] = b11 * dq1 + b12 * dq2 + b13 * dq3;
}

SMAC_DEV bool bc_has(const BcRegion &r, int j, int k)
{
    return r.ibcval == 31 ? j == r.jbeg && k >= r.kbeg && k <= r.kend
                          : k == r.kbeg && j >= r.jbeg && j <= r.jend;
}

// Block (x, y) takes BC_THREADS points of region y.  A point's first region applies all of its
// regions, in file order.
template <typename LT>
SMAC_DEV void b_bc(const Blk &bk, const Dims &d, const BcTable &t, double pout, double alpha,
                   double beta, const DevStats *__restrict__ st, const double *__restrict__ x,
                   const double *__restrict__ y, const double *__restrict__ met,
                   const double *__restrict__ q, double *__restrict__ s, LT *btc, LT *bjm,
                   LT *bjp, LT *bkm, LT *bkp)
{
    const int i0 = (int)bk.y, n = (int)(bk.x * BC_THREADS + threadIdx.x);
    const bool column = t.r[i0].ibcval == 31;
    const int j = t.r[i0].jbeg + (column ? 0 : n), k = t.r[i0].kbeg + (column ? n : 0);
    if (!bc_has(t.r[i0], j, k)) return;
    for (int i = 0; i < i0; ++i)
        if (bc_has(t.r[i], j, k)) return;
    const double clift = st->clift;
    for (int i = i0; i < t.n; ++i) {
        if (!bc_has(t.r[i], j, k)) continue;
        const int ib = t.r[i].ibcval;
        if (ib == 31) bc_outj<LT>(d, j, k, pout, q, s, btc, bjm, bjp);
        else if (ib == 0) bc_noslk<LT>(d, j, k, q, s, btc, bkp);
        else if (ib == 25) bc_cgridk<LT>(d, j, k, alpha, beta, clift, x, y, met, q, s, btc, bkm);
    }
}

// the grid of a table: the longest region's points, the regions
static dim3 bc_grid(const BcTable &t)
{
    int most = 1;
    for (int i = 0; i < t.n; ++i) {
        const BcRegion &r = t.r[i];
        const int n = r.ibcval == 31 ? r.kend - r.kbeg + 1 : r.jend - r.jbeg + 1;
        most = n > most ? n : most;
    }
    return dim3((unsigned)((most + BC_THREADS - 1) / BC_THREADS), (unsigned)t.n);
}

template <typename LT>
__global__ void __launch_bounds__(BC_THREADS)
k_bc(Dims d, BcTable t, double pout, double alpha, double beta, const DevStats *__restrict__ st,
     const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ met,
     const double *__restrict__ q, double *__restrict__ s, LT *btc, LT *bjm, LT *bjp, LT *bkm,
     LT *bkp)
{
    b_bc<LT>(hw_blk(), d, t, pout, alpha, beta, st, x, y, met, q, s, btc, bjm, bjp, bkm, bkp);
}

// ---------------------------------------------------------------------------------------
// resid + rhsnorm: isamax over s*dj (ties to the first index, ref/blas.f:48-83) for all 3N
// entries and for the first N, and sum of s^2; partials per block, then one final block.
// The partition is fixed, so the result is the same on every run.  945x241: 6 us for the partials
// (1.2 TB/s; with a 64-bit remainder for every value 11-12 us beside the SA) and 4.6 us for the
// final block, both mostly a launch and the latency of one round of loads.

struct ArgMax {
    double v;
    long i;
};

SMAC_DEV ArgMax amax_join(ArgMax a, ArgMax b)
{
    if (b.v > a.v || (b.v == a.v && b.i < a.i)) return b;
    return a;
}

constexpr int RED_THREADS = 256;

// Thread 0 gets the block's values: t joins t + w, w = 128, 64 .. 1, the last 64 in one wave.
SMAC_DEV void red_tree(ArgMax &all, ArgMax &first, double &ss)
{
    constexpr int W = 64;
    static_assert(RED_THREADS == 4 * W, "two steps through LDS");
    __shared__ double v[2 * W][3];
    __shared__ long id[2 * W][2];
    const int t = threadIdx.x;
    for (int w = RED_THREADS / 2; w >= W; w >>= 1) {
        if (t >= w && t < 2 * w) {
            v[t - w][0] = all.v; id[t - w][0] = all.i;
            v[t - w][1] = first.v; id[t - w][1] = first.i;
            v[t - w][2] = ss;
        }
        __syncthreads();
        if (t < w) {
            all = amax_join(all, {v[t][0], id[t][0]});
            first = amax_join(first, {v[t][1], id[t][1]});
            ss = ss + v[t][2];
        }
        __syncthreads();
    }
    if (t >= W) return;
    for (int w = W / 2; w > 0; w >>= 1) {
        all = amax_join(all, {__shfl_down(all.v, w), __shfl_down(all.i, w)});
        first = amax_join(first, {__shfl_down(first.v, w), __shfl_down(first.i, w)});
        ss = ss + __shfl_down(ss, w);
    }
}

SMAC_DEV void b_resid_partial(const Blk &bk, Dims d, const double *__restrict__ s,
                              const double *__restrict__ dj, double *__restrict__ part_v,
                              long *__restrict__ part_i, double *__restrict__ part_s)
{
    const long N = d.N, n3 = 3 * N;
    ArgMax all = {-1.0, 0x7fffffffffffffffL}, first = {-1.0, 0x7fffffffffffffffL};
    double ss = 0.0;
    for (long i = (long)bk.x * blockDim.x + threadIdx.x; i < n3;
         i += (long)bk.nx * blockDim.x) {
        const long p = i < N ? i : i < 2 * N ? i - N : i - 2 * N;
        double sv = s[i];
        double a = fabs(sv * dj[p]);
        all = amax_join(all, {a, i});
        if (i < N) first = amax_join(first, {a, i});
        ss += sv * sv;
    }
    const int t = threadIdx.x;
    red_tree(all, first, ss);
    if (t == 0) {
        part_v[2 * bk.x] = all.v; part_i[2 * bk.x] = all.i;
        part_v[2 * bk.x + 1] = first.v; part_i[2 * bk.x + 1] = first.i;
        part_s[bk.x] = ss;
    }
}

__global__ void __launch_bounds__(RED_THREADS)
k_resid_partial(Dims d, const double *__restrict__ s, const double *__restrict__ dj,
                double *__restrict__ part_v, long *__restrict__ part_i, double *__restrict__ part_s)
{
    b_resid_partial(hw_blk(), d, s, dj, part_v, part_i, part_s);
}

SMAC_DEV void b_resid_final(const Dims &d, int nparts, int nt, double beta,
                            const double *__restrict__ s, const double *__restrict__ dj,
                            const double *__restrict__ part_v, const long *__restrict__ part_i,
                            const double *__restrict__ part_s, DevStats *st)
{
    const int t = threadIdx.x;
    ArgMax all = {-1.0, 0x7fffffffffffffffL}, first = {-1.0, 0x7fffffffffffffffL};
    double ss = 0.0;
    for (int b = t; b < nparts; b += RED_THREADS) {
        all = amax_join(all, {part_v[2 * b], part_i[2 * b]});
        first = amax_join(first, {part_v[2 * b + 1], part_i[2 * b + 1]});
        ss += part_s[b];
    }
    red_tree(all, first, ss);
    if (t == 0) {
        const long N = d.N;
        long irmax = all.i;                  // 0-based index into the 3N array
        long id = first.i;
        int bad = 0;
        // an all-NaN residual leaves no candidate: report it instead of indexing with it
        if (irmax < 0 || irmax >= 3 * N) { irmax = 0; bad = 1; }
        if (id < 0 || id >= N) { id = 0; bad = 1; }
        long p = irmax % N;
        st->kres = (int)(p / d.jm) + 1;
        st->jres = (int)(p % d.jm) + 1;
        st->resmax = fabs(s[irmax] * dj[p]);
        if (nt == 1) {
            st->resmax0 = st->resmax;
            if (st->resmax0 < 1.) st->resmax0 = 1.0;
        }
        st->divmax = fabs(s[id] * dj[id] / beta);
        st->rhsnorm = sqrt(ss);
        st->nonfinite = bad || !(st->rhsnorm <= 1.0e300);
    }
}

__global__ void __launch_bounds__(RED_THREADS)
k_resid_final(Dims d, int nparts, int nt, double beta, const double *__restrict__ s,
              const double *__restrict__ dj, const double *__restrict__ part_v,
              const long *__restrict__ part_i, const double *__restrict__ part_s, DevStats *st)
{
    b_resid_final(d, nparts, nt, beta, s, dj, part_v, part_i, part_s, st);
}

// ---------------------------------------------------------------------------------------
// launchers

template <typename LT>
void launch_assemble(hipStream_t sm, const Dims &d, const DevParams &prm, const double *q,
                     const double *met, const double *dj, double *s, LT *btc, LT *bjm, LT *bjp,
                     LT *bkm, LT *bkp)
{
    const int rows = asm_rows(d);
    dim3 blk(64), grd((d.jm + ASM_COLS - 1) / ASM_COLS, (d.km + rows - 1) / rows);
    hipLaunchKernelGGL(k_assemble<LT>, grd, blk, 0, sm, d, prm, rows, q, met, dj, s, btc, bjm, bjp,
                       bkm, bkp);
}

template <typename LT>
void launch_bc(hipStream_t sm, const Dims &d, const DevParams &prm, const BcRegion *regs,
               int nreg, const DevStats *st, const double *x, const double *y, const double *met,
               const double *q, double *s, LT *btc, LT *bjm, LT *bjp, LT *bkm, LT *bkp)
{
    // up to BC_MAX regions per launch; more go in further launches, still in file order
    BcTable t{};
    for (int i = 0; i <= nreg; ++i) {
        if (i == nreg || t.n == BC_MAX) {
            if (t.n)
                hipLaunchKernelGGL(k_bc<LT>, bc_grid(t), dim3(BC_THREADS), 0, sm, d, t, prm.pout,
                                   prm.alpha, prm.beta, st, x, y, met, q, s, btc, bjm, bjp, bkm,
                                   bkp);
            t.n = 0;
            if (i == nreg) break;
        }
        const int ib = regs[i].ibcval;
        if (ib != 31 && ib != 0 && ib != 25) continue;   // wake cuts: bcimpds in the solve
        t.r[t.n++] = regs[i];
    }
}

void launch_resid(hipStream_t sm, const Dims &d, int nt, double beta, const double *s,
                  const double *dj, Scratch &w, DevStats *st)
{
    int nb = w.nred;
    hipLaunchKernelGGL(k_resid_partial, dim3(nb), dim3(RED_THREADS), 0, sm, d, s, dj, w.red_v,
                       w.red_i, w.red_s);
    hipLaunchKernelGGL(k_resid_final, dim3(1), dim3(RED_THREADS), 0, sm, d, nb, nt, beta, s, dj,
                       w.red_v, w.red_i, w.red_s, st);
}

// ---- multi-case launches ------------------------------------------------------------------

template <typename LT>
AsmArgs asm_args(const Dims &d, const DevParams &prm, const double *q, const double *met,
                 const double *dj, double *s, LT *btc, LT *bjm, LT *bjp, LT *bkm, LT *bkp)
{
    // the cases of a batch fill the chip together
    constexpr int rows = 4;
    return AsmArgs{(unsigned)((d.jm + ASM_COLS - 1) / ASM_COLS), (unsigned)((d.km + rows - 1) / rows),
                   d, prm, rows, q, met, dj, s, btc, bjm, bjp, bkm, bkp};
}

template <typename LT>
void bc_args(const Dims &d, const DevParams &prm, const BcRegion *regs, int nreg,
             const DevStats *st, const double *x, const double *y, const double *met,
             const double *q, double *s, LT *btc, LT *bjm, LT *bjp, LT *bkm, LT *bkp,
             std::vector<BcArgs> &out)
{
    BcTable t{};
    for (int i = 0; i <= nreg; ++i) {
        if (i == nreg || t.n == BC_MAX) {
            if (t.n) {
                const dim3 g = bc_grid(t);
                out.push_back(BcArgs{g.x, g.y, d, t, prm.pout, prm.alpha, prm.beta, st, x, y, met,
                                     q, s, btc, bjm, bjp, bkm, bkp});
            }
            t.n = 0;
            if (i == nreg) break;
        }
        const int ib = regs[i].ibcval;
        if (ib != 31 && ib != 0 && ib != 25) continue;
        t.r[t.n++] = regs[i];
    }
}

ResidPArgs residp_args(const Dims &d, const double *s, const double *dj, Scratch &w)
{
    return ResidPArgs{(unsigned)w.nred, 1u, d, s, dj, w.red_v, w.red_i, w.red_s};
}

ResidFArgs residf_args(const Dims &d, int nt, double beta, const double *s, const double *dj,
                       Scratch &w, DevStats *st)
{
    return ResidFArgs{1u, 1u, d, w.nred, nt, beta, s, dj, w.red_v, w.red_i, w.red_s, st};
}

template <typename LT>
struct CAssemble {
    using Args = AsmArgs;
    static constexpr int THREADS = 64, WAVES = 2;
    static SMAC_DEV void run(const Blk &b, const Args &a)
    {
        b_assemble<LT>(b, a.rows, a.d, a.prm, as_global(a.q), as_global(a.met), as_global(a.dj),
                       as_global(a.s), (LT *)as_global(a.btc), (LT *)as_global(a.bjm),
                       (LT *)as_global(a.bjp), (LT *)as_global(a.bkm), (LT *)as_global(a.bkp));
    }
};

template <typename LT>
struct CBc {
    using Args = BcArgs;
    static constexpr int THREADS = BC_THREADS;
    static SMAC_DEV void run(const Blk &b, const Args &a)
    {
        b_bc<LT>(b, a.d, a.t, a.pout, a.alpha, a.beta, as_global(a.st), as_global(a.x),
                 as_global(a.y), as_global(a.met), as_global(a.q), as_global(a.s),
                 (LT *)as_global(a.btc), (LT *)as_global(a.bjm), (LT *)as_global(a.bjp),
                 (LT *)as_global(a.bkm), (LT *)as_global(a.bkp));
    }
};

struct CResidP {
    using Args = ResidPArgs;
    static constexpr int THREADS = RED_THREADS;
    static SMAC_DEV void run(const Blk &b, const Args &a)
    {
        b_resid_partial(b, a.d, as_global(a.s), as_global(a.dj), as_global(a.part_v),
                        as_global(a.part_i), as_global(a.part_s));
    }
};

struct CResidF {
    using Args = ResidFArgs;
    static constexpr int THREADS = RED_THREADS;
    static SMAC_DEV void run(const Blk &, const Args &a)
    {
        b_resid_final(a.d, a.nparts, a.nt, a.beta, as_global(a.s), as_global(a.dj),
                      as_global(a.part_v), as_global(a.part_i), as_global(a.part_s),
                      as_global(a.st));
    }
};

template <class C>
static void multi_launch(hipStream_t sm, const MultiTab<typename C::Args> &t)
{
    if (t.n > 0 && t.nblk > 0)
        hipLaunchKernelGGL(k_multi<C>, dim3(t.nblk), dim3(C::THREADS), 0, sm, t.args, t.start, t.n,
                           t.item_case, t.active);
}

template <typename LT> void multi_assemble(hipStream_t sm, const MultiTab<AsmArgs> &t)
{
    multi_launch<CAssemble<LT>>(sm, t);
}
template <typename LT> void multi_bc(hipStream_t sm, const MultiTab<BcArgs> &t)
{
    multi_launch<CBc<LT>>(sm, t);
}
void multi_resid_partial(hipStream_t sm, const MultiTab<ResidPArgs> &t) { multi_launch<CResidP>(sm, t); }
void multi_resid_final(hipStream_t sm, const MultiTab<ResidFArgs> &t) { multi_launch<CResidF>(sm, t); }

template AsmArgs asm_args<double>(const Dims &, const DevParams &, const double *, const double *,
                                  const double *, double *, double *, double *, double *,
                                  double *, double *);
template AsmArgs asm_args<float>(const Dims &, const DevParams &, const double *, const double *,
                                 const double *, double *, float *, float *, float *, float *,
                                 float *);
template void bc_args<double>(const Dims &, const DevParams &, const BcRegion *, int,
                              const DevStats *, const double *, const double *, const double *,
                              const double *, double *, double *, double *, double *, double *,
                              double *, std::vector<BcArgs> &);
template void bc_args<float>(const Dims &, const DevParams &, const BcRegion *, int,
                             const DevStats *, const double *, const double *, const double *,
                             const double *, double *, float *, float *, float *, float *,
                             float *, std::vector<BcArgs> &);
template void multi_assemble<double>(hipStream_t, const MultiTab<AsmArgs> &);
template void multi_assemble<float>(hipStream_t, const MultiTab<AsmArgs> &);
template void multi_bc<double>(hipStream_t, const MultiTab<BcArgs> &);
template void multi_bc<float>(hipStream_t, const MultiTab<BcArgs> &);

template void launch_assemble<double>(hipStream_t, const Dims &, const DevParams &,
                                      const double *, const double *, const double *, double *,
                                      double *, double *, double *, double *, double *);
template void launch_assemble<float>(hipStream_t, const Dims &, const DevParams &,
                                     const double *, const double *, const double *, double *,
                                     float *, float *, float *, float *, float *);
template void launch_bc<double>(hipStream_t, const Dims &, const DevParams &, const BcRegion *,
                                int, const DevStats *, const double *, const double *,
                                const double *, const double *, double *, double *, double *,
                                double *, double *, double *);
template void launch_bc<float>(hipStream_t, const Dims &, const DevParams &, const BcRegion *, int,
                               const DevStats *, const double *, const double *, const double *,
                               const double *, double *, float *, float *, float *, float *,
                               float *);

}  // namespace smac
