// Block line relaxation of the implicit iteration: lrelax / ljsweep / lksweep
// (ref/lrelax.f:51-561), the 3x3 block-tridiagonal Crout factor and its undo (btlu3j,
// btlu3k, btund3j; ref/btlu3.f:52-838) and the wake-cut injection after every sweep
// (bcimpds single-rank branch, ref/bc.f:571-591).
//
// Reference order ("parity mode"): the xi sweep visits k-lines in Gauss-Seidel order
// (line k reads dq of line k-1 from the same sweep), so lines are strictly sequential.  One
// workgroup walks the lines: one wavefront runs the block forward/back substitution with the
// factored blocks, the others form the updates and the next line's right-hand side behind it.
// The factorisations are independent per line: one lane per line.
#include "smac_dev.h"
#include "smac_kernels.h"

#include <type_traits>

namespace smac {

// 3x3 helpers on registers, entry (m,n) at index m + 3n ------------------------------------

template <typename T>
SMAC_DEV void lu3(T b[9])
{
    // ref/btlu3.f:148-155
    b[0] = (T)1. / b[0];
    b[3] = b[3] * b[0];
    b[6] = b[6] * b[0];
    b[4] = (T)1. / (b[4] - b[1] * b[3]);
    b[7] = (b[7] - b[1] * b[6]) * b[4];
    b[5] = b[5] - b[2] * b[3];
    b[8] = (T)1. / (b[8] - b[2] * b[6] - b[7] * b[5]);
}

template <typename T>
SMAC_DEV void csolve3(const T b[9], T c[9])
{
    // c <- b^-1 c, column by column (ref/btlu3.f:157-179)
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        T d1 = b[0] * c[3 * n];
        T d2 = b[4] * (c[1 + 3 * n] - b[1] * d1);
        T d3 = b[8] * (c[2 + 3 * n] - b[2] * d1 - b[5] * d2);
        c[2 + 3 * n] = d3;
        c[1 + 3 * n] = d2 - b[7] * c[2 + 3 * n];
        c[3 * n] = d1 - b[6] * c[2 + 3 * n] - b[3] * c[1 + 3 * n];
    }
}

template <typename T>
SMAC_DEV void bminus3(T b[9], const T a[9], const T c[9])
{
    // b <- b - a c (ref/btlu3.f:245-273)
#pragma unroll
    for (int n = 0; n < 3; ++n)
#pragma unroll
        for (int m = 0; m < 3; ++m)
            b[m + 3 * n] = b[m + 3 * n] - a[m] * c[3 * n] - a[m + 3] * c[1 + 3 * n] -
                           a[m + 6] * c[2 + 3 * n];
}

template <typename T>
SMAC_DEV void bplus3(T b[9], const T a[9], const T c[9])
{
    // b <- b + a c (ref/btlu3.f:660-690)
#pragma unroll
    for (int n = 0; n < 3; ++n)
#pragma unroll
        for (int m = 0; m < 3; ++m)
            b[m + 3 * n] = b[m + 3 * n] + a[m] * c[3 * n] + a[m + 3] * c[1 + 3 * n] +
                           a[m + 6] * c[2 + 3 * n];
}

template <typename T>
SMAC_DEV void unlu3(T b[9])
{
    // recompose a factored block (ref/btlu3.f:640-650)
    b[8] = (T)1. / b[8] + b[2] * b[6] + b[5] * b[7];
    b[5] = b[5] + b[2] * b[3];
    b[4] = (T)1. / b[4];
    b[7] = b[7] * b[4] + b[1] * b[6];
    b[4] = b[4] + b[1] * b[3];
    b[0] = (T)1. / b[0];
    b[6] = b[6] * b[0];
    b[3] = b[3] * b[0];
}

template <typename T>
SMAC_DEV void ctimes3(const T b[9], T c[9])
{
    // c <- b c (ref/btlu3.f:700-735)
    T t[9];
#pragma unroll
    for (int n = 0; n < 3; ++n)
#pragma unroll
        for (int m = 0; m < 3; ++m)
            t[m + 3 * n] = b[m] * c[3 * n] + b[m + 3] * c[1 + 3 * n] + b[m + 6] * c[2 + 3 * n];
#pragma unroll
    for (int e = 0; e < 9; ++e) c[e] = t[e];
}

template <typename LT>
SMAC_DEV void ld9(const LT *__restrict__ a, long N, long p, LT r[9])
{
#pragma unroll
    for (int e = 0; e < 9; ++e) r[e] = a[e * N + p];
}
template <typename LT>
SMAC_DEV void st9(LT *__restrict__ a, long N, long p, const LT r[9])
{
#pragma unroll
    for (int e = 0; e < 9; ++e) a[e * N + p] = r[e];
}

// ------------------------------------------------------------------------------------------
// the factored lines, packed: block b of line l (its points 16b .. 16b+15, q = point in the
// block, c = equation) is one chunk of 4096 bytes, as the chain of a sweep reads it:
//   [q][c][16 B]  (a_c0 a_c1), (a_c2 f8)       lower band of equation c
//   [q][16 B]     (f0 f1) (f2 f3) (f4 f5) (f6 f7)   factored diagonal
//   [q][c][16 B]  (C_c0 C_c1), (C_c2 -)        factored upper band
// a is zero at a line's first point and C at its last, whose terms the reference does not form
// (they meet a zero there); past the line's end everything is zero.

typedef double v2d __attribute__((ext_vector_type(2)));
constexpr int RB = 16, RCHUNK = 4096;
constexpr int RA0 = 0, RA1 = 768, RD = 1536, RC0 = 2560, RC1 = 3328;

SMAC_DEV int ref_blocks(int len) { return (len + RB - 1) / RB; }
SMAC_DEV char *ref_point(char *pk, int len, int l, int i)   // + q*48 or q*16 by the caller
{
    return pk + ((long)l * ref_blocks(len) + i / RB) * RCHUNK;
}

long lr_ref_bytes(const Dims &d)
{
    const long xi = (long)d.km * ((d.jm + RB - 1) / RB), eta = (long)d.jm * ((d.km + RB - 1) / RB);
    return (xi > eta ? xi : eta) * RCHUNK;
}

// factorisation along lines: btlu3j (lines of constant k, walking j) and btlu3k, one lane per
// line, into the packed chunks.  `stride` is the point step along the line, `lstride` the step
// between lines.  A point's recurrence takes about 0.4 us (three dependent divisions); its 27
// values are loaded PF points ahead, since a load on the chain would cost three times that
// (119x31, xi lines: 190 us without, 103 us with and a line per wave).
template <typename LT>
__global__ void __launch_bounds__(64) k_btlu3(long N, int nline, int len, long stride,
                                             long lstride, const LT *__restrict__ a,
                                             const LT *__restrict__ b, const LT *__restrict__ c,
                                             char *__restrict__ pk)
{
    constexpr int PF = 4;
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= nline) return;
    LT la[PF][9], lb[PF][9], lc[PF][9];
    auto load = [&](int u, int i) {
        const long p = lstride * l + stride * (i < len ? i : len - 1);
        ld9(b, N, p, lb[u]);
        ld9(a, N, p, la[u]);
        ld9(c, N, p, lc[u]);
    };
#pragma unroll
    for (int u = 0; u < PF; ++u) load(u, u);
    LT cp[9];
#pragma unroll
    for (int e = 0; e < 9; ++e) cp[e] = (LT)0;
    auto put = [&](int i, const LT *aa, const LT *bb, const LT *cc) {
        const int q = i % RB;
        char *ch = ref_point(pk, len, l, i);
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            char *lane = ch + q * 48 + m * 16;
            *(v2d *)(lane + RA0) = v2d{aa[m], aa[m + 3]};
            *(v2d *)(lane + RA1) = v2d{aa[m + 6], bb[8]};
            *(v2d *)(lane + RC0) = v2d{cc[m], cc[m + 3]};
            *(v2d *)(lane + RC1) = v2d{cc[m + 6], 0.};
        }
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *(v2d *)(ch + RD + g * 256 + q * 16) = v2d{bb[2 * g], bb[2 * g + 1]};
    };
    for (int i0 = 0; i0 < len; i0 += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int i = i0 + u;
            if (i >= len) break;
            if (i > 0) {
                bminus3(lb[u], la[u], cp);
            } else {
#pragma unroll
                for (int e = 0; e < 9; ++e) la[u][e] = (LT)0;
            }
            lu3(lb[u]);
            csolve3(lb[u], lc[u]);
            if (i == len - 1) {
#pragma unroll
                for (int e = 0; e < 9; ++e) lc[u][e] = (LT)0;
            }
#pragma unroll
            for (int e = 0; e < 9; ++e) cp[e] = lc[u][e];
            put(i, la[u], lb[u], lc[u]);
            load(u, i + PF);
        }
    }
#pragma unroll
    for (int e = 0; e < 9; ++e) cp[e] = (LT)0;
    for (int i = len; i < ref_blocks(len) * RB; ++i) put(i, cp, cp, cp);
}

// btund3j: recompose btc and bjp from their xi factors (ref/btlu3.f:628-838), one point per
// thread (the factors are in the chunks, so a point does not wait for its neighbours)
template <typename LT>
__global__ void __launch_bounds__(256) k_btund3(long N, int len, const LT *__restrict__ a,
                                               LT *__restrict__ b, LT *__restrict__ c,
                                               const char *__restrict__ pk)
{
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const int l = (int)(p / len), i = (int)(p % len);
    auto band = [&](int ii, LT o[9]) {   // C of point ii
        const char *ch = ref_point((char *)pk, len, l, ii) + ii % RB * 48;
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const v2d t = *(const v2d *)(ch + m * 16 + RC0);
            o[m] = t.x;
            o[m + 3] = t.y;
            o[m + 6] = *(const double *)(ch + m * 16 + RC1);
        }
    };
    LT bb[9];
    {
        const char *ch = ref_point((char *)pk, len, l, i);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const v2d t = *(const v2d *)(ch + RD + g * 256 + i % RB * 16);
            bb[2 * g] = t.x;
            bb[2 * g + 1] = t.y;
        }
        bb[8] = ((const double *)(ch + i % RB * 48 + RA1))[1];
    }
    unlu3(bb);
    if (i < len - 1) {
        LT cc[9];
        band(i, cc);
        ctimes3(bb, cc);
        st9(c, N, p, cc);
    }
    if (i > 0) {
        LT aa[9], cp[9];
        ld9(a, N, p, aa);
        band(i - 1, cp);
        bplus3(bb, aa, cp);
    }
    st9(b, N, p, bb);
}

// ------------------------------------------------------------------------------------------
// one sweep in reference line order (ljsweep / lksweep): lines one after another in one
// workgroup; `eta` chooses xi lines (lines of constant k) or eta lines (constant j).
//
// Wave 0 is the chain: forward substitution along the line, then back.  Lane 4q + c holds
// equation c of point q of a block of 16 points (c = 3 repeats c = 2), so a block's operands
// are six loads for the wave; the points are then solved one after another by all lanes, the
// one whose turn it is for good, and its result goes to the next through scalar registers
// (v_readlane).  A forward step is 21 FP64 operations (33 where one lane does all three
// equations), a backward one 6, with no LDS access or load in either.
// Waves 1..SW take segments of 64 points: as soon as the chain has passed a segment on its way
// back, they form the under-relaxed update there and the next line's right-hand side, whose
// operands they loaded while the chain was running.  The waves meet in LDS counters, each wait
// for a wave that does not wait back: the chain for a segment's right-hand side of its line,
// a segment for the chain's blocks of the line before.
//
// What bounds it: the chain, two dependent block steps per point, line after line: about 65 ns
// each (21 and 6 FP64 operations and the passing on, at the 5 cycles a lone wavefront takes per
// instruction).  At 119x31 a sweep takes 480 us; with one lane solving all three equations out
// of LDS, and every line's operands staged and its right-hand side formed between the chains,
// it took 1050 us (xi) and 1380 us (eta).
constexpr int SW = 7;

__global__ void __launch_bounds__(64 * (SW + 1))
k_sweep_ref(Dims d, int eta, int nsweep, double underr, double *__restrict__ dq,
            const double *__restrict__ s, const char *__restrict__ pk,
            const double *__restrict__ om, const double *__restrict__ op)
{
    // om/op: blocks to the neighbouring lines (bkm/bkp for xi, bjm/bjp for eta)
    extern __shared__ double line[];   // per point 3: right-hand side, then y, then x
    const long N = d.N;
    const int nline = eta ? d.jm : d.km;
    const int len = eta ? d.km : d.jm;
    const long stride = eta ? d.jm : 1;          // along a line
    const long lstride = eta ? 1 : d.jm;         // between lines
    const bool rev = (nsweep / 2) * 2 == nsweep;
    const int nblk = ref_blocks(len), nseg = (len + 63) / 64;
    int *back = (int *)(line + 3 * nblk * RB);   // backward blocks done, over all lines
    int *ready = back + 1;                       // per segment: lines whose right-hand side is there
    auto ld = [](const int *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    auto st = [](int *p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    for (int i = 3 * len + threadIdx.x; i < 3 * nblk * RB; i += 64 * (SW + 1)) line[i] = 0.;
    for (int i = threadIdx.x; i < 1 + nseg; i += 64 * (SW + 1)) back[i] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto line_of = [&](int ll) { return rev ? nline - 1 - ll : ll; };

    if (wave > 0) {
        const double half = 0.5;
        // the update of the line just solved (l, -1: none yet), then the right-hand side of the next
        // (ln, -1: none), with x and y the dq of the lines on its two sides
        for (int ll = -1; ll < nline; ++ll) {
            const int l = ll < 0 ? -1 : line_of(ll), ln = ll + 1 < nline ? line_of(ll + 1) : -1;
            const int lmn = ln - 1 > 0 ? ln - 1 : 0;
            const int lpl = ln + 1 < nline - 1 ? ln + 1 : nline - 1;
            const double rkm = (double)(float)(ln - lmn - 1);
            const double rkp = (double)(float)(lpl - ln - 1);
            const double swm = half + copysign(half, rkm);
            const double swp = half + copysign(half, rkp);
            // bring the chunks of the line after next closer (the chain loads them from L2)
            int warm = 0;
            if (ll + 2 < nline) {
                const char *w = pk + (long)line_of(ll + 2) * nblk * RCHUNK;
                for (int o = ((wave - 1) * 64 + lane) * 128; o < nblk * RCHUNK; o += SW * 64 * 128)
                    warm ^= *(const int *)(w + o);
            }
            for (int sg = nseg - 1 - ((nseg - wave) % SW + SW) % SW; sg >= 0; sg -= SW) {
                const int i = sg * 64 + lane;
                const bool in = i < len;
                const long po = stride * (in ? i : 0);
                double dl[3], sn[3], x[3], y[3], bo[9], bp[9];
                if (l >= 0) {
#pragma unroll
                    for (int n = 0; n < 3; ++n) dl[n] = dq[n * N + lstride * l + po];
                }
                if (ln >= 0) {
                    const long p = lstride * ln + po;
#pragma unroll
                    for (int n = 0; n < 3; ++n) {
                        sn[n] = s[n * N + p];
                        x[n] = lmn == l ? 0. : dq[n * N + lstride * lmn + po];
                        y[n] = lpl == l ? 0. : dq[n * N + lstride * lpl + po];
                    }
                    ld9(om, N, p, bo);
                    ld9(op, N, p, bp);
                }
                if (l >= 0) {
                    const int need = ll * nblk + nblk - 4 * sg;
                    while (ld(back) < need) __builtin_amdgcn_s_sleep(1);
                    asm volatile("" ::: "memory");
                    if (in) {
#pragma unroll
                        for (int n = 0; n < 3; ++n) {
                            const double v = dl[n] + underr * (line[3 * i + n] - dl[n]);
                            dq[n * N + lstride * l + po] = v;
                            x[n] = lmn == l ? v : x[n];
                            y[n] = lpl == l ? v : y[n];
                        }
                    }
                }
                if (ln >= 0) {
                    if (in) {
#pragma unroll
                        for (int m = 0; m < 3; ++m) {
                            double bm = bo[m] * x[0] + bo[m + 3] * x[1] + bo[m + 6] * x[2];
                            double bq = bp[m] * y[0] + bp[m + 3] * y[1] + bp[m + 6] * y[2];
                            line[3 * i + m] = sn[m] - bm * swm - bq * swp;
                        }
                    }
                    asm volatile("" ::: "memory");
                    st(&ready[sg], ll + 2);
                }
            }
            asm volatile("" : : "v"(warm));
        }
        return;
    }

    // ---- the chain
    const int q = lane >> 2, c = (lane & 3) < 2 ? lane & 3 : 2;
    const int o3 = q * 48 + c * 16, o1 = q * 16;
    struct Fwd { v2d a0, a1, f[4]; } F[2];
    struct Bck { v2d c0; double c2; } B[3];
    auto ldf = [&](Fwd &t, const char *ch) {
        t.a0 = *(const v2d *)(ch + RA0 + o3);
        t.a1 = *(const v2d *)(ch + RA1 + o3);
#pragma unroll
        for (int g = 0; g < 4; ++g) t.f[g] = *(const v2d *)(ch + RD + g * 256 + o1);
    };
    auto ldb = [&](Bck &t, const char *ch) {
        t.c0 = *(const v2d *)(ch + RC0 + o3);
        t.c2 = *(const double *)(ch + RC1 + o3);
    };
    auto chunk = [&](int l, int b) {
        b = b < 0 ? 0 : (b < nblk ? b : nblk - 1);
        return pk + ((long)l * nblk + b) * RCHUNK;
    };
    auto quad_value = [](double v, auto C) {   // v of lane C of the quad
        const unsigned long long u = (unsigned long long)__double_as_longlong(v);
        constexpr int ctrl = decltype(C)::value * 0x55;
        const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)u, ctrl, 0xf, 0xf, false);
        const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(u >> 32), ctrl, 0xf, 0xf, false);
        return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                                (unsigned long long)(unsigned)lo));
    };
    auto lane_value = [](double v, int from) {
        const unsigned long long u = (unsigned long long)__double_as_longlong(v);
        const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, from);
        const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), from);
        return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    };
    ldf(F[0], chunk(line_of(0), 0));
    ldf(F[1], chunk(line_of(0), 1));
    for (int ll = 0; ll < nline; ++ll) {
        const int l = line_of(ll);
#pragma unroll
        for (int u = 0; u < 3; ++u) ldb(B[u], chunk(l, nblk - 1 - u));
        // forward with the factored diagonal blocks and the lower band (ref/lrelax.f:331-351)
        double r1 = 0., r2 = 0., r3 = 0.;   // the point before, in every lane
        auto forward = [&](const Fwd &t, int b) {
            if (b % 4 == 0) {
                while (ld(&ready[b / 4]) < ll + 1) {}
                asm volatile("" ::: "memory");
            }
            double *slot = line + 3 * (b * RB + q) + c;
            const double rhs = *slot;
            const double b0 = t.f[0].x, b1 = t.f[0].y, b2 = t.f[1].x, b3 = t.f[1].y, b4 = t.f[2].x,
                         b5 = t.f[2].y, b6 = t.f[3].x, b7 = t.f[3].y, b8 = t.a1.y;
            double y1 = 0., y2 = 0., y3 = 0.;   // this lane's point, once its turn has come
#pragma unroll
            for (int g = 0; g < RB; ++g) {
                const double tt = rhs - t.a0.x * r1 - t.a0.y * r2 - t.a1.x * r3;
                const double t1 = quad_value(tt, std::integral_constant<int, 0>{}),
                             t2 = quad_value(tt, std::integral_constant<int, 1>{}),
                             t3 = quad_value(tt, std::integral_constant<int, 2>{});
                if (q == g) {
                    const double d1 = b0 * t1;
                    const double d2 = b4 * (t2 - b1 * d1);
                    const double d3 = b8 * (t3 - b2 * d1 - b5 * d2);
                    y3 = d3;
                    y2 = d2 - b7 * y3;
                    y1 = d1 - b6 * y3 - b3 * y2;
                }
                r1 = lane_value(y1, 4 * g);
                r2 = lane_value(y2, 4 * g);
                r3 = lane_value(y3, 4 * g);
            }
            *slot = c == 0 ? y1 : c == 1 ? y2 : y3;
        };
        for (int b = 0;;) {
            forward(F[0], b);
            if (++b == nblk) break;
            ldf(F[0], chunk(l, b + 1));
            forward(F[1], b);
            if (++b == nblk) break;
            ldf(F[1], chunk(l, b + 1));
        }
        if (ll + 1 < nline) {
            ldf(F[0], chunk(line_of(ll + 1), 0));
            ldf(F[1], chunk(line_of(ll + 1), 1));
        }
        // back substitution with the upper band (ref/lrelax.f:367-373)
        double x1 = 0., x2 = 0., x3 = 0.;   // the point after, in every lane
        auto backward = [&](const Bck &t, int b) {
            double *slot = line + 3 * (b * RB + q) + c;
            double v = *slot;
#pragma unroll
            for (int g = RB - 1; g >= 0; --g) {
                const double tt = v - t.c0.x * x1 - t.c0.y * x2 - t.c2 * x3;
                v = q == g ? tt : v;
                x1 = lane_value(tt, 4 * g);
                x2 = lane_value(tt, 4 * g + 1);
                x3 = lane_value(tt, 4 * g + 2);
            }
            *slot = v;
            asm volatile("" ::: "memory");
            st(back, ll * nblk + nblk - b);
        };
        for (int b = nblk - 1;;) {
            backward(B[0], b);
            if (--b < 0) break;
            ldb(B[0], chunk(l, b - 2));
            backward(B[1], b);
            if (--b < 0) break;
            ldb(B[1], chunk(l, b - 2));
            backward(B[2], b);
            if (--b < 0) break;
            ldb(B[2], chunk(l, b - 2));
        }
    }
}

// wake-cut injection, bcimpds single-rank branch (ref/bc.f:571-591): k = 0 row of the cut.
// Pairs whose indices fall outside the row are skipped.
SMAC_DEV void b_wake(const Blk &bk, long N, int jm, int neqs, int npair, int base,
                     const int *__restrict__ pairs, const double *__restrict__ sq,
                     double *__restrict__ ds, double *__restrict__ rhs)
{
    const int i = bk.x * blockDim.x + threadIdx.x;
    if (i >= npair) return;
    const long jt = pairs[2 * i] - base, jb = pairs[2 * i + 1] - base;
    if (jt < 0 || jt >= jm || jb < 0 || jb >= jm) return;
    for (int n = 0; n < neqs; ++n) {
        double snew = 0.5 * (sq[n * N + jt + jm] + sq[n * N + jb + jm]);
        double dsnew = 0.5 * (ds[n * N + jt + jm] + ds[n * N + jb + jm]);
        ds[n * N + jt] = snew + dsnew - sq[n * N + jt];
        rhs[n * N + jt] = ds[n * N + jt];
    }
}

__global__ void k_wake(long N, int jm, int neqs, int npair, int base,
                       const int *__restrict__ pairs, const double *__restrict__ sq,
                       double *__restrict__ ds, double *__restrict__ rhs)
{
    b_wake(hw_blk(), N, jm, neqs, npair, base, pairs, sq, ds, rhs);
}

__global__ void k_fill(double *__restrict__ a, long n, double v)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long)gridDim.x * blockDim.x)
        a[i] = v;
}

WakeArgs wake_args(const Dims &d, int neqs, const WakePairs &w, const double *sq, double *ds,
                   double *rhs)
{
    return WakeArgs{(unsigned)(w.n > 0 ? (w.n + 63) / 64 : 0), 1u, d.N, d.jm, neqs, w.n, w.base,
                    w.pairs, sq, ds, rhs};
}

struct CWake {
    using Args = WakeArgs;
    static constexpr int THREADS = 64;
    static SMAC_DEV void run(const Blk &b, const Args &a)
    {
        b_wake(b, a.N, a.jm, a.neqs, a.npair, a.base, as_global(a.pairs), as_global(a.sq),
               as_global(a.ds), as_global(a.rhs));
    }
};

void multi_wake(hipStream_t sm, const MultiTab<WakeArgs> &t)
{
    if (t.n > 0 && t.nblk > 0)
        hipLaunchKernelGGL(k_multi<CWake>, dim3(t.nblk), dim3(64), 0, sm, t.args, t.start, t.n,
                           t.item_case, t.active);
}

void launch_wake(hipStream_t sm, const Dims &d, int neqs, const WakePairs &w, const double *sq,
                 double *ds, double *rhs)
{
    if (w.n <= 0) return;
    hipLaunchKernelGGL(k_wake, dim3((w.n + 63) / 64), dim3(64), 0, sm, d.N, d.jm, neqs, w.n,
                       w.base, w.pairs, sq, ds, rhs);
}

void launch_lrelax_ref(hipStream_t sm, const Dims &d, const DevParams &prm, int njsp, int nksp,
                       int nbcimp, const WakePairs &w, const double *q, double *dq, double *s,
                       double *btc, const double *bjm, double *bjp, const double *bkm,
                       const double *bkp, void *pack)
{
    const long N = d.N;
    char *pk = (char *)pack;
    // lines per workgroup of the factor kernels (one lane per line): as few as leave a wave per
    // SIMD -- the lanes of a wave load from as many cache lines (31 lines of 119 points: 160 us
    // in one wave, 103 us in 31)
    auto lines = [](int nline) { return (unsigned)((nline + 1023) / 1024); };
    auto groups = [&](int nline) { return (nline + lines(nline) - 1) / lines(nline); };
    auto sweep = [&](int eta, int ns, const double *om, const double *op) {
        const int len = eta ? d.km : d.jm;
        const size_t lds = sizeof(double) * 3 * ((len + RB - 1) / RB * RB) + 4 * (1 + (len + 63) / 64);
        hipLaunchKernelGGL(k_sweep_ref, dim3(1), dim3(64 * (SW + 1)), lds, sm, d, eta, ns, prm.underr,
                           dq, s, pk, om, op);
        if ((ns / nbcimp) * nbcimp == ns) launch_wake(sm, d, 3, w, q, dq, s);
    };
    hipLaunchKernelGGL(k_fill, dim3(256), dim3(256), 0, sm, dq, 3 * N, 0.0);
    if (njsp > 0)
        hipLaunchKernelGGL(k_btlu3<double>, dim3(groups(d.km)), dim3(lines(d.km)), 0, sm, N, d.km,
                           d.jm, 1L, (long)d.jm, bjm, btc, bjp, pk);
    for (int nj = 1; nj <= njsp; ++nj) sweep(0, nj, bkm, bkp);
    if (njsp > 0)
        hipLaunchKernelGGL(k_btund3<double>, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, sm, N,
                           d.jm, bjm, btc, bjp, pk);
    if (nksp > 0)
        hipLaunchKernelGGL(k_btlu3<double>, dim3(groups(d.jm)), dim3(lines(d.jm)), 0, sm, N, d.jm,
                           d.km, (long)d.jm, 1L, bkm, btc, bkp, pk);
    for (int nk = 1; nk <= nksp; ++nk) sweep(1, nk, bjm, bjp);
}

}  // namespace smac
