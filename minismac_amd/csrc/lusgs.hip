// LU-SGS of the implicit iteration: lusgs / lusini3 / lusini1 (ref/lusgs.f:51-236) and the
// approximate factorisation solve (D+L) D^-1 (D+U) of ilusol3 / ilusol1 (ref/ilusol.f).
//
// The reference sweeps in natural order (j fastest).  Point (j,k) of the forward sweep reads
// only (j-1,k) and (j,k-1) -- plus (jmax,k-1) at j = 1 and (jmax,kmax)/(1,kmax) at j = jmax
// in the backward sweep, through blocks that the C-grid boundary rows leave exactly zero
// (bjm at j = 1, bjp at j = jmax; ref/bc.f:1622-1648 after the blanking of ref/step.f:386-413)
// -- so visiting the hyperplanes h = j+k in order performs the reference's arithmetic
// operation for operation.
//
// Schedule on gfx950:
//  1. k_shear: the block planes and the right-hand side are gathered into the workspace by
//     hyperplanes: the operands of 16 rows (64 for the scalar system) of one hyperplane are one
//     contiguous chunk.  The diagonal factors (lusini3 / lusini1) are formed on the way.
//  2. k_band (forward): the rows are cut into bands, one workgroup each, whose computing
//     wavefront walks the hyperplanes upward.  (j-1,k) is its own result of the previous step
//     (registers), (j,k-1) the previous lane's (a DPP shift).
//  3. k_mid: the middle step, pointwise (not for FP32-LHS, whose scaled form needs none).
//  4. k_band (backward): the mirror image, h downward, bands handing their first row down.
//  5. k_unshear: dq (and, for callers that want it, the middle-step rhs) back to the natural
//     layout; then the wake-cut rows (bcimpds) as in the reference.
// Every point performs the reference's expressions in the reference's order.  The terms the
// reference does not form (at the first/last row or column) have their blocks stored as zeros
// and meet neighbour values that are zero, so they leave the sum as it is.
#include "smac_dev.h"
#include "smac_kernels.h"

#include <type_traits>
#include <utility>

namespace smac {

constexpr unsigned long long EDGE_EMPTY = 0x7ff4dead0000beefull;   // signalling NaN

// A slot word counts as not yet written when its high half is the sentinel's: a hand-over
// value is finite, so its high half never is (0x7ff4dead is a NaN exponent), and a word read
// while it was being written, with the sentinel's high half and the value's low half, is
// then waited for and read again instead of taken as a NaN.
SMAC_DEV bool edge_empty(unsigned long long v)
{
    return (unsigned)(v >> 32) == (unsigned)(EDGE_EMPTY >> 32);
}

constexpr int EDGE_SPIN_MAX = 1000000;
constexpr int BAND_LANES = 64;
constexpr int HP0 = 16;          // empty hyperplanes before h = 0 and after h = H
constexpr int EPAD = 128;        // padding slots on either side of a band's edge row

// ------------------------------------------------------------------------------------------
// the workspace layout
//
// The sweep of a band is a chain of one step per hyperplane, so what a step costs is what one
// wavefront issues in it.  The 3x3 system therefore gives a row to four lanes instead of one:
// lane 4q + c holds equation c of row q (c = 3 repeats c = 2), forms that equation's 6 products
// and differences, and the three sums are exchanged inside the quad (DPP) for the 3x3
// substitution, which every lane then performs.  A step of 16
// rows issues about 70 instructions where one row per lane took over 130, it needs 4 KB of
// operands instead of 15, and its operand reads are 8 LDS reads instead of 15.
//
// A chunk is what one step of 16 rows reads, as the lanes read it (FP64; c = equation):
//   groups of 768 bytes [q][c][16 B]:  (jn0 jn1) (jn2 kn0) (kn1 kn2) of equation c, (r_c f8)
//   groups of 256 bytes [q][16 B]:     (f0 f1) (f2 f3) (f4 f5) (f6 f7)
// jn, kn: the blocks to the j- and the k-neighbour (bjm, bkm forward; bjp, bkp backward).  The
// backward chunk holds only the first three groups: r and the factors are the forward chunk's,
// where the forward sweep and the middle step leave their results in r's place, and the
// backward sweep dq.  FP32-LHS (scaled form, no factors): two groups, (jn0 jn1 jn2 r_c) and
// (kn0 kn1 kn2 -), in both chunks; the forward sweep's result goes to the backward chunk's r.
// The scalar system: 64 rows, (jn kn) [row][16 B] and (r f) [row][16 B], the backward chunk
// only the first.
template <int NEQ, typename T> struct Form;
template <> struct Form<3, double> {
    static constexpr int ROWS = 16, FB = 4096, BB = 2304;   // rows; bytes of a chunk: fwd, bwd
    static constexpr int IMG = 4096, BOWN = 2304;   // a step's operands; those of the bwd chunk
    static constexpr int RG = 2304, RS = 48, RC = 16, RO = 0;   // r_c of row q: RG + q*RS + c*RC + RO
    static constexpr int RING = 24, FLY = 4;       // steps in the LDS ring; in flight per loader
    static constexpr int SUB = 4;                   // steps between two looks at the counters
    static constexpr int AHEAD = 2;                 // steps the LDS reads run ahead
    static constexpr bool Y_BWD = false;            // forward result into the backward chunk
    static constexpr int SKEW = 0;                  // steps that four rows run behind the four before
    static constexpr int EDGE = 4;                  // words of a step's hand-over values
};
template <> struct Form<3, float> {
    static constexpr int ROWS = 16, FB = 1536, BB = 1536;
    static constexpr int IMG = 1536, BOWN = 1536;
    static constexpr int RG = 0, RS = 48, RC = 16, RO = 12;
    // more in flight (FLY) and the loaders, who count a step as landed FLY of their steps later,
    // run out of ring: 11 323 -> 330 us a pass, 13 486; 7 or a longer ring gains nothing
    static constexpr int RING = 48, FLY = 9;
    static constexpr int SUB = 4;
    static constexpr int AHEAD = 2;
    static constexpr bool Y_BWD = true;
    static constexpr int SKEW = AHEAD;
    static constexpr int EDGE = 20;
};
template <> struct Form<1, double> {
    static constexpr int ROWS = 64, FB = 2048, BB = 1024;
    static constexpr int IMG = 2048, BOWN = 1024;
    static constexpr int RG = 1024, RS = 16, RC = 0, RO = 0;
    static constexpr int RING = 36, FLY = 6;
    static constexpr int SUB = 4;
    static constexpr int AHEAD = 2;
    static constexpr bool Y_BWD = false;
    static constexpr int SKEW = 0;
    static constexpr int EDGE = 1;
};

// The forms of large launches (see band_form for the rule).  FormMost: a shorter ring, of which
// four fit a compute unit's 160 KB instead of two.
template <int NEQ, typename T> struct FormMany;
template <> struct FormMany<3, float> : Form<3, float> {
    static constexpr int RING = 36, FLY = 6;
};
template <> struct FormMany<1, double> : Form<1, double> {
    static constexpr int RING = 18, FLY = 4, SUB = 2;
};
struct FormMost : Form<3, float> {
    static constexpr int RING = 24, FLY = 4;
};

// the forward / backward chunk of rows tile*ROWS.. of hyperplane h
template <class F> SMAC_DEV char *fwd_chunk(const LusgsWs &w, int h, int tile)
{
    return (char *)w.lhs + ((long)(h + HP0) * (w.ks / F::ROWS) + tile) * F::FB;
}
template <class F> SMAC_DEV char *bwd_chunk(const LusgsWs &w, int h, int tile)
{
    const long nt = w.ks / F::ROWS;
    return (char *)w.lhs + (long)(w.H + 1 + 2 * HP0) * nt * F::FB + ((long)(h + HP0) * nt + tile) * F::BB;
}
// r of equation c of row k (0..ROWS-1) of the chunk at p
template <class F> SMAC_DEV char *r_of(char *p, int k, int c)
{
    return p + F::RG + k * F::RS + c * F::RC + F::RO;
}

// ------------------------------------------------------------------------------------------
// diagonal factors

template <typename LT>
SMAC_DEV void lu_factor3(const LT t[9], LT f[9])
{
    // lusini3 (ref/lusgs.f:196-209), entry (m,n) at m + 3n
    f[0] = (LT)1. / t[0];
    f[3] = t[3] * f[0];
    f[6] = t[6] * f[0];
    f[1] = t[1];
    f[4] = (LT)1. / (t[4] - f[1] * f[3]);
    f[7] = (t[7] - f[1] * f[6]) * f[4];
    f[2] = t[2];
    f[5] = t[5] - f[2] * f[3];
    f[8] = (LT)1. / (t[8] - f[2] * f[6] - f[5] * f[7]);
}

template <typename AT>
SMAC_DEV void lu_solve3(const AT f[9], AT r1, AT r2, AT r3, AT o[3])
{
    // forward/back substitution with the lusini3 factors (ref/ilusol.f:146-170)
    AT z1 = r1 * f[0];
    AT z2 = (r2 - f[1] * z1) * f[4];
    AT z3 = (r3 - f[2] * z1 - f[5] * z2) * f[8];
    o[2] = z3;
    o[1] = z2 - f[7] * o[2];
    o[0] = z1 - f[6] * o[2] - f[3] * o[1];
}

// FP32-LHS form of the 3x3 substitution (fused multiply-adds; not the reference's rounding)
SMAC_DEV void lu_solve3_fma(const float f[9], float r1, float r2, float r3, float o[3])
{
    const float z1 = r1 * f[0];
    const float z2 = __builtin_fmaf(-f[1], z1, r2) * f[4];
    const float z3 = __builtin_fmaf(-f[5], z2, __builtin_fmaf(-f[2], z1, r3)) * f[8];
    o[2] = z3;
    o[1] = __builtin_fmaf(-f[7], o[2], z2);
    o[0] = __builtin_fmaf(-f[3], o[1], __builtin_fmaf(-f[6], o[2], z1));
}

// ------------------------------------------------------------------------------------------
// natural <-> chunk layout: a workgroup takes 16 hyperplanes x ROWS rows.  Threads read the
// planes with 16 consecutive j of a row side by side (128 bytes), build the chunks in LDS and
// copy them out whole, contiguously.  Bound by HBM: at 1889x481 FP64 it reads 349 MB and
// writes 363 MB in 163 us (4.4 TB/s; tiles of the natural planes with partly written lines and
// 464 bytes a point took 215 us), at 945x241 34 us (was 48).

constexpr int TH = 16, TILE_THREADS = 256;
template <class F> constexpr int OVER = 8 + 3 * F::SKEW;   // steps past a band's ends, at most
constexpr int IMG_PAD = 16;      // bytes between the tile's chunks in LDS: the 16 hyperplanes of
                                 // one row land in different banks

SMAC_DEV void copy_out(const unsigned char *img, char *dst, int nh, int bytes, int stride,
                       long pitch)
{
    const int per = bytes / 16;
    for (int e = threadIdx.x; e < nh * per; e += TILE_THREADS) {
        const int hh = e / per, o = (e - hh * per) * 16;
        *(uint4 *)(dst + hh * pitch + o) = *(const uint4 *)(img + hh * stride + o);
    }
}

template <typename LT, int NEQ>
SMAC_DEV void b_shear(const Blk &bk, const Dims &d, const LusgsWs &w,
                      const double *__restrict__ rhs, const LT *__restrict__ btc,
                      const LT *__restrict__ bjm, const LT *__restrict__ bkm,
                      const LT *__restrict__ bjp, const LT *__restrict__ bkp, LT *__restrict__ fac)
{
    using F = Form<NEQ, LT>;
    constexpr int STR = F::FB + IMG_PAD;
    __shared__ __attribute__((aligned(16))) unsigned char img[TH * STR];
    {
        // hand-over slots of both sweeps: the jm real ones become the sentinel, the padding
        // on either side stays a finite value (the dummy region after them is not touched)
        const long nthr = (long)bk.nx * bk.ny * TILE_THREADS;
        const long t0 = ((long)bk.y * bk.nx + bk.x) * TILE_THREADS + threadIdx.x;
        const long nreal = 2L * w.nband * w.epitch;
        for (long i = t0; i < nreal; i += nthr) {
            const long pos = (i % w.epitch) / 4;
            w.edge[i] = (pos >= EPAD && pos < EPAD + d.jm) ? EDGE_EMPTY : 0ull;
        }
    }
    // the tiles the sweeps may touch: they run less than OVER steps past a band's ends (those
    // chunks are reset to zeros too), and a band of fewer rows may reach over a tile's edge
    const int tile = bk.y, k0 = tile * F::ROWS, h0 = (int)bk.x * TH - HP0;
    const int over = OVER<F> + (w.rows == F::ROWS ? 0 : F::ROWS);
    if (h0 + TH <= k0 - over || h0 > d.jm + k0 + F::ROWS + over) return;
    const int nh = w.H + HP0 + 1 - h0 < TH ? w.H + HP0 + 1 - h0 : TH;   // hyperplanes of the tile
    const long fpitch = (long)(w.ks / F::ROWS) * F::FB, bpitch = (long)(w.ks / F::ROWS) * F::BB;
    const int hh = threadIdx.x % TH;
    unsigned char *im = img + hh * STR;
    char *fdst = fwd_chunk<F>(w, h0, tile), *bdst = bwd_chunk<F>(w, h0, tile);
    constexpr int PTS = TH * F::ROWS / TILE_THREADS;   // points per thread
    constexpr int NB = NEQ * NEQ;
    if constexpr (NEQ == 3) {
        static_assert(PTS == 1, "one point per thread");
        const int kk = threadIdx.x / TH, k = k0 + kk, j = h0 + hh - k;
        const bool in = k < d.km && j >= 0 && j < d.jm;
        const long p = P(d, j, k);
        LT t[9], f[9], jm[9], km[9], jp[9], kp[9], r[3];
        // the blocks of terms the reference does not form are stored as zeros
        const bool hjm = in && j > 0, hkm = in && k > 0, hjp = in && j < d.jm - 1,
                   hkp = in && k < d.km - 1;
#pragma unroll
        for (int m = 0; m < 9; ++m) {
            t[m] = in ? btc[m * d.N + p] : (LT)0;
            jm[m] = hjm ? bjm[m * d.N + p] : (LT)0;
            km[m] = hkm ? bkm[m * d.N + p] : (LT)0;
            jp[m] = hjp ? bjp[m * d.N + p] : (LT)0;
            kp[m] = hkp ? bkp[m * d.N + p] : (LT)0;
        }
#pragma unroll
        for (int m = 0; m < 3; ++m) r[m] = in ? (LT)rhs[m * d.N + p] : (LT)0;
        lu_factor3<LT>(t, f);
#pragma unroll
        for (int m = 0; m < 9; ++m) {
            if (fac && in) fac[m * d.N + p] = f[m];
            f[m] = in ? f[m] : (LT)0;
        }
        if constexpr (sizeof(LT) == 8) {
            typedef double v2 __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                unsigned char *a = im + kk * 48 + c * 16;
                *(v2 *)(a) = v2{jm[c], jm[c + 3]};
                *(v2 *)(a + 768) = v2{jm[c + 6], km[c]};
                *(v2 *)(a + 1536) = v2{km[c + 3], km[c + 6]};
                *(v2 *)(a + 2304) = v2{r[c], f[8]};
            }
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *(v2 *)(im + 3072 + g * 256 + kk * 16) = v2{f[2 * g], f[2 * g + 1]};
            __syncthreads();
            copy_out(img, fdst, nh, F::FB, STR, fpitch);
            __syncthreads();
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                unsigned char *a = im + kk * 48 + c * 16;
                *(v2 *)(a) = v2{jp[c], jp[c + 3]};
                *(v2 *)(a + 768) = v2{jp[c + 6], kp[c]};
                *(v2 *)(a + 1536) = v2{kp[c + 3], kp[c + 6]};
            }
        } else {
            // The FP32-LHS sweeps use the scaled form of the same operator: with D = LU(btc),
            // (D+L) y = r is y = D^-1 r - (D^-1 L) y, and (D+U) x = D y is x = y - (D^-1 U) x,
            // so the four neighbour blocks and the rhs are stored premultiplied by D^-1 (three
            // substitutions per block), and neither the sweeps nor the middle step need the
            // factors.
            typedef float v4 __attribute__((ext_vector_type(4)));
            auto scale = [&](LT *b, int cols) {
                for (int c = 0; c < cols; ++c) {
                    float o[3];
                    lu_solve3_fma(f, b[3 * c], b[3 * c + 1], b[3 * c + 2], o);
                    b[3 * c] = o[0];
                    b[3 * c + 1] = o[1];
                    b[3 * c + 2] = o[2];
                }
            };
            scale(jm, 3);
            scale(km, 3);
            scale(jp, 3);
            scale(kp, 3);
            scale(r, 1);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                unsigned char *a = im + kk * 48 + c * 16;
                *(v4 *)(a) = v4{jm[c], jm[c + 3], jm[c + 6], r[c]};
                *(v4 *)(a + 768) = v4{km[c], km[c + 3], km[c + 6], 0.f};
            }
            __syncthreads();
            copy_out(img, fdst, nh, F::FB, STR, fpitch);
            __syncthreads();
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                unsigned char *a = im + kk * 48 + c * 16;
                *(v4 *)(a) = v4{jp[c], jp[c + 3], jp[c + 6], 0.f};
                *(v4 *)(a + 768) = v4{kp[c], kp[c + 3], kp[c + 6], 0.f};
            }
        }
    } else {
        typedef double v2 __attribute__((ext_vector_type(2)));
        double jp[PTS], kp[PTS];
#pragma unroll
        for (int i = 0; i < PTS; ++i) {
            const int kk = threadIdx.x / TH + i * (TILE_THREADS / TH), k = k0 + kk, j = h0 + hh - k;
            const bool in = k < d.km && j >= 0 && j < d.jm;
            const long p = P(d, j, k);
            const double f = in ? 1. / btc[p] : 0.;   // lusini1 (ref/lusgs.f:230-234)
            if (fac && in) fac[p] = f;
            *(v2 *)(im + kk * 16) = v2{in && j > 0 ? bjm[p] : 0., in && k > 0 ? bkm[p] : 0.};
            *(v2 *)(im + 1024 + kk * 16) = v2{in ? rhs[p] : 0., f};
            jp[i] = in && j < d.jm - 1 ? bjp[p] : 0.;
            kp[i] = in && k < d.km - 1 ? bkp[p] : 0.;
        }
        __syncthreads();
        copy_out(img, fdst, nh, F::FB, STR, fpitch);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PTS; ++i)
            *(v2 *)(im + (threadIdx.x / TH + i * (TILE_THREADS / TH)) * 16) = v2{jp[i], kp[i]};
    }
    __syncthreads();
    copy_out(img, bdst, nh, F::BB, STR, bpitch);
}

template <typename LT, int NEQ>
__global__ void __launch_bounds__(TILE_THREADS)
k_shear(Dims d, LusgsWs w, const double *__restrict__ rhs, const LT *__restrict__ btc,
        const LT *__restrict__ bjm, const LT *__restrict__ bkm, const LT *__restrict__ bjp,
        const LT *__restrict__ bkp, LT *__restrict__ fac)
{
    b_shear<LT, NEQ>(xcd_blk(), d, w, rhs, btc, bjm, bkm, bjp, bkp, fac);
}

// the grid of k_shear: hyperplanes -HP0 .. H + HP0, the rows' tiles
template <typename LT, int NEQ> static dim3 shear_grid(const Dims &d, const LusgsWs &w)
{
    using F = Form<NEQ, LT>;
    return dim3((unsigned)((w.H + 1 + 2 * HP0 + TH - 1) / TH),
                (unsigned)((d.km + F::ROWS - 1) / F::ROWS));
}

// The wake-cut injection (bcimpds, ref/bc.f:571-591) of the points that a workgroup of k_unshear
// writes, on the way: a cut point's new value follows from its pair's dq on the second row, which
// the workspace holds.  A launch of its own behind k_unshear cost 4 us: 945x241 FP32-LHS passes 323
// -> 319 us, 119x31 laminar steps 113 -> 111.
struct WakeIn {
    WakePairs pairs;
    const double *sq;
    double *rhs;          // gets the cut points' values too
};

// r's place in the forward chunks (dq after the backward sweep, the middle-step rhs before
// it; FP32-LHS has the latter in the backward chunks) -> natural FP64 planes
template <int NEQ, typename T>
SMAC_DEV void b_unshear(const Blk &bk, const Dims &d, const LusgsWs &w, bool mid,
                        double *__restrict__ dst, const WakeIn &wk)
{
    using F = Form<NEQ, T>;
    constexpr int UK = 16;                  // rows per workgroup
    __shared__ T lds[NEQ][UK][TH + 1];
    const int k0 = bk.y * UK, h0 = bk.x * TH;
    if (h0 + TH <= k0 || h0 >= d.jm + k0 + UK) return;
    const int tile = k0 / F::ROWS, kt = k0 % F::ROWS;
    for (int e = threadIdx.x; e < TH * UK * NEQ; e += TILE_THREADS) {
        const int hh = e / (UK * NEQ), o = e - hh * (UK * NEQ), kk = o / NEQ, c = o - kk * NEQ;
        char *ch = mid && F::Y_BWD ? bwd_chunk<F>(w, h0 + hh, tile) : fwd_chunk<F>(w, h0 + hh, tile);
        lds[c][kk][hh] = *(const T *)r_of<F>(ch, kt + kk, c);
    }
    // the pair of each point on the first row
    const bool cut = k0 == 0 && wk.pairs.n > 0;
    __shared__ int pair[TH];
    if (cut) {
        if (threadIdx.x < TH) pair[threadIdx.x] = -1;
        __syncthreads();
        for (int i = threadIdx.x; i < wk.pairs.n; i += TILE_THREADS) {
            const long jt = wk.pairs.pairs[2 * i] - wk.pairs.base, jb = wk.pairs.pairs[2 * i + 1] - wk.pairs.base;
            if (jt < 0 || jt >= d.jm || jb < 0 || jb >= d.jm) continue;
            if (jt >= h0 && jt < h0 + TH) pair[jt - h0] = (int)jb;
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < TH * UK; e += TILE_THREADS) {
        const int kk = e / TH, hh = e % TH, k = k0 + kk, j = h0 + hh - k;
        if (j < 0 || j >= d.jm || k >= d.km) continue;
        const long p = P(d, j, k);
        const int jb = cut && k == 0 ? pair[hh] : -1;
        if (jb >= 0) {
            // the second row's points of columns j and jb
            char *ct = fwd_chunk<F>(w, j + 1, 0), *cb = fwd_chunk<F>(w, jb + 1, 0);
#pragma unroll
            for (int m = 0; m < NEQ; ++m) {
                const double snew = 0.5 * (wk.sq[m * d.N + j + d.jm] + wk.sq[m * d.N + jb + d.jm]);
                const double dsnew = 0.5 * ((double)*(const T *)r_of<F>(ct, 1, m) +
                                            (double)*(const T *)r_of<F>(cb, 1, m));
                const double v = snew + dsnew - wk.sq[m * d.N + j];
                dst[m * d.N + p] = v;
                wk.rhs[m * d.N + p] = v;
            }
            continue;
        }
#pragma unroll
        for (int m = 0; m < NEQ; ++m) dst[m * d.N + p] = (double)lds[m][kk][hh];
    }
}

template <int NEQ, typename T>
__global__ void __launch_bounds__(TILE_THREADS)
k_unshear(Dims d, LusgsWs w, bool mid, double *__restrict__ dst, WakeIn wk)
{
    b_unshear<NEQ, T>(xcd_blk(), d, w, mid, dst, wk);
}

static dim3 unshear_grid(const Dims &d, const LusgsWs &w)
{
    return dim3((unsigned)((w.H + TH) / TH), (unsigned)((d.km + 15) / 16));
}

// ------------------------------------------------------------------------------------------
// middle step: rhs <- D rhs, pointwise (ref/ilusol.f:307-341 for neqs = 3; ref/ilusol.f:548-556
// for neqs = 1, where D = 1/b)

template <typename LT, int NEQ>
SMAC_DEV void b_mid(const Blk &bk, const Dims &d, const LusgsWs &w)
{
    if constexpr (sizeof(LT) == 8) {
        using F = Form<NEQ, LT>;
        typedef double v2 __attribute__((ext_vector_type(2)));
        for (long i = (long)bk.x * blockDim.x + threadIdx.x; i < (long)(w.H + 1) * w.ks;
             i += (long)bk.nx * blockDim.x) {
            const int h = (int)(i / w.ks), k = (int)(i % w.ks), j = h - k;
            if (k >= d.km || j < 0 || j >= d.jm) continue;
            char *ch = fwd_chunk<F>(w, h, k / F::ROWS);
            const int kk = k % F::ROWS;
            if constexpr (NEQ == 3) {
                v2 *R0 = (v2 *)r_of<F>(ch, kk, 0), *R1 = (v2 *)r_of<F>(ch, kk, 1),
                   *R2 = (v2 *)r_of<F>(ch, kk, 2);
                double f[9];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const v2 t = *(const v2 *)(ch + 3072 + g * 256 + kk * 16);
                    f[2 * g] = t.x;
                    f[2 * g + 1] = t.y;
                }
                const v2 r0 = *R0;
                f[8] = r0.y;
                const double o0 = r0.x, o1 = R1->x, o2 = R2->x, one = 1.;
                double b11 = one / f[0];
                double b12 = f[3] * b11;
                double b13 = f[6] * b11;
                double b21 = f[1];
                double b22 = one / f[4] + f[1] * f[3];
                double b23 = f[7] / f[4] + f[1] * f[6];
                double b31 = f[2];
                double b32 = f[5] + f[2] * f[3];
                double b33 = one / f[8] + f[2] * f[6] + f[5] * f[7];
                R0->x = b11 * o0 + b12 * o1 + b13 * o2;
                R1->x = b21 * o0 + b22 * o1 + b23 * o2;
                R2->x = b31 * o0 + b32 * o1 + b33 * o2;
            } else {
                v2 *R = (v2 *)r_of<F>(ch, kk, 0);
                const v2 t = *R;
                R->x = t.x / t.y;
            }
        }
    }
}

template <typename LT, int NEQ>
__global__ void __launch_bounds__(256) k_mid(Dims d, LusgsWs w)
{
    b_mid<LT, NEQ>(hw_blk(), d, w);
}

template <int NEQ> static unsigned mid_blocks(const LusgsWs &w)
{
    const long nb = ((long)(w.H + 1) * w.ks + 255) / 256;
    return (unsigned)(nb > 4096 ? 4096 : nb);
}

// ------------------------------------------------------------------------------------------
// band sweeps
//
// A band's workgroup has a computing wavefront, LOADERS loaders and a hand-over wavefront:
//  - the loaders stream the steps' operands into an LDS ring (LDS DMA, no registers), up to
//    RING steps ahead of the computing wavefront, and count the steps that have landed;
//  - the hand-over wavefront polls the slots that the neighbour band writes (its boundary
//    row's results, through device memory) and counts the steps it has copied into LDS;
//  - the computing wavefront reads a coming step's operands from LDS under this step's
//    arithmetic, and every SUB steps looks at the counters and publishes its progress.
// They meet only in these counters (no barrier in the steps); each wait is for a wave that
// does not wait back, so they end: a loader waits for the computing wave's progress, the
// computing wave for the counters, and the hand-over wave, whose polls are bounded (on
// time-out it raises the stall flag and hands zeros on), for the band before, which was
// dispatched earlier and finds a place whatever other launches hold (band_form).
//
// What bounds a sweep: its chain of jmax + kmax - 1 steps, each as long as the computing
// wavefront takes to issue it -- a wavefront alone on its SIMD issues one VALU instruction
// per 5 cycles (measured), so about 68 instructions FP64 make 144 ns, 22 FP32 60 ns -- and the
// hand-over lag of 2 us per band beyond the 16 rows' own skew.  The hand-over wavefront shares
// the computing one's SIMD, which therefore runs at a higher priority (with four polls in flight,
// as once: backward sweep 218 -> 209 us, an LU-SGS solve at 477x121 253.5 -> 250; now 204 and 242).
//
// The FP32 step has no 3x3 substitution, so what it issued was mostly moves: three results
// broadcast in the quad, each passed to the next row by two moves (one inside a row of 16 lanes,
// one across), and selects.  Its fused multiply-adds now take the quad's values themselves; a
// lane passes its own equation on with one move; and across the rows of 16 lanes, which have no
// such move for four lanes at once, a result goes through LDS with the hand-over values: four
// rows run SKEW steps behind the four before, 90 more steps at 945x241.  A pass there 347 -> 324
// us, each sweep 112 -> 105.  FP64 keeps the moves: it would save 4 of 68 instructions and pay
// 8% more steps.
//
// At 945x241 the forward sweep takes 211 us FP64, 105 us FP32 and 64 us for the scalar system;
// with one row per lane, 64-row bands and an s_barrier per step it took 318, 215 and 130-150 us (whose step moved 15 KB
// through one CU, next to 51 FP64 operations in every lane); at 1889x481 848 -> 438 us FP64.
constexpr int LOADERS = 3;       // loader wavefronts, each taking every third step
constexpr int BAND_WAVES = 2 + LOADERS;

// Hand-over slots are read and written with the agent-coherent cache policy (sc1), the form
// the compiler gives relaxed agent-scope atomics; every slot is an aligned 8-byte word.
constexpr int EDGE_POLICY = 0x10;

using rsrc_t = __amdgpu_buffer_rsrc_t;
typedef unsigned int v2u __attribute__((ext_vector_type(2)));

// raw buffer over `bytes` bytes (gfx9 resource word 3); stores beyond it are dropped
SMAC_DEV rsrc_t mk_rsrc(const void *p, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes,
                                             0x00020000);
}

// Slots are written one 8-byte word per store and lane.  A buffer store of more than 8 bytes
// whose offset comes from an SGPR can read its data registers after the next instruction has
// issued, and the compiler does not keep that instruction off them.
SMAC_DEV void edge_st(unsigned lo, unsigned hi, rsrc_t r, unsigned vo, unsigned so)
{
    __builtin_amdgcn_raw_buffer_store_b64(v2u{lo, hi}, r, (int)vo, (int)so, EDGE_POLICY);
}

// gfx9 s_waitcnt immediate: wait until at most n vector-memory operations are outstanding
constexpr int vmcnt_imm(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }

SMAC_DEV void dma16(const char *src, unsigned char *lds)
{
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                     (__attribute__((address_space(3))) void *)lds, 16, 0, 0);
}

// DPP moves of a 32- or 64-bit value; lanes that receive nothing keep `old`
template <int CTRL, int ROWS, int BANKS> SMAC_DEV float dpp(float old, float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old),
                                                                 __builtin_bit_cast(int, v), CTRL,
                                                                 ROWS, BANKS, false));
}
template <int CTRL, int ROWS, int BANKS> SMAC_DEV double dpp(double old, double v)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned long long w = (unsigned long long)__double_as_longlong(old);
    const int lo = __builtin_amdgcn_update_dpp((int)(unsigned)w, (int)(unsigned)u, CTRL, ROWS, BANKS,
                                               false);
    const int hi = __builtin_amdgcn_update_dpp((int)(unsigned)(w >> 32), (int)(unsigned)(u >> 32),
                                               CTRL, ROWS, BANKS, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                            (unsigned long long)(unsigned)lo));
}

// v of the row before; the first row receives `in`.  3x3: rows are quads of lanes, so the last
// quad of a DPP row of 16 lanes passes to the next one (row_bcast:15), the others by row_shr:4.
template <int NEQ, typename T> SMAC_DEV T from_row_before(T v, T in)
{
    if constexpr (NEQ == 3) return dpp<0x114, 0xf, 0xe>(dpp<0x142, 0xe, 0x1>(in, v), v);
    else return dpp<0x138, 0xf, 0xf>(in, v);   // wave_shr:1
}
// v of lane C of the quad
template <int C> SMAC_DEV float quad_lane(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), C * 0x55,
                                                              0xf, 0xf, false));
}
template <int C> SMAC_DEV double quad_lane(double v)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)u, C * 0x55, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(u >> 32), C * 0x55, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                            (unsigned long long)(unsigned)lo));
}

// Forces x to be computed where it stands.
template <typename T>
SMAC_DEV T keep(T x)
{
    asm volatile("" : "+v"(x));
    return x;
}

// the words of a hand-over slot: the FP64 value, or the FP32 one with a zero high half
SMAC_DEV void slot_word(double v, unsigned &lo, unsigned &hi)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    lo = (unsigned)u;
    hi = (unsigned)(u >> 32);
}
SMAC_DEV void slot_word(float v, unsigned &lo, unsigned &hi)
{
    lo = __builtin_bit_cast(unsigned, v);
    hi = 0u;
}
SMAC_DEV void slot_value(unsigned long long e, double &v) { v = __longlong_as_double((long long)e); }
SMAC_DEV void slot_value(unsigned long long e, float &v)
{
    v = __builtin_bit_cast(float, (unsigned)e);
}

// one lane's operands of a step
template <int NEQ, typename T> struct Ops {
    T jn[3], kn[3], r, f[9];
    T e[sizeof(T) == 4 ? 1 : NEQ];   // the incoming hand-over values (FP32: of this lane's equation)
};

// the shared state of a band's waves
template <class F, typename T> struct BandLds {
    __attribute__((aligned(16))) T edge[F::RING][F::EDGE];   // the hand-over values
    __attribute__((aligned(16))) int cnt[4];   // steps landed (loaders), steps handed over
    int consumed;       // steps whose ring slots are free again
    __attribute__((aligned(16))) unsigned char ring[F::RING * F::IMG];
};
SMAC_DEV int cnt_ld(const int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
SMAC_DEV void cnt_st(int *p, int v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The loader's counter accesses, as asm: the compiler makes any LDS access of a wave with LDS
// DMA in flight wait for all of it (over twice the time of a step).
SMAC_DEV unsigned lds_addr(const void *p)
{
    return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}
SMAC_DEV int cnt_ld_dma(unsigned a)
{
    int v;
    asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(a) : "memory");
    return __builtin_amdgcn_readfirstlane(v);
}
SMAC_DEV void cnt_st_dma(unsigned a, int v)   // every lane stores the same word
{
    asm volatile("ds_write_b32 %0, %1" : : "v"(a), "v"(v) : "memory");
}

// reads a step's operands from the ring: lane base `b` and the row base `rb` (3x3 FP64
// factors) of slot SLOT; immediate offsets
template <int NEQ, typename T>
SMAC_DEV void read_ops(Ops<NEQ, T> &o, const unsigned char *b, const unsigned char *rb,
                       const T *e)
{
    if constexpr (NEQ == 3 && sizeof(T) == 8) {
        typedef double v2 __attribute__((ext_vector_type(2)));
        const v2 a0 = *(const v2 *)b, a1 = *(const v2 *)(b + 768), a2 = *(const v2 *)(b + 1536),
                 a3 = *(const v2 *)(b + 2304);
        o.jn[0] = a0.x;
        o.jn[1] = a0.y;
        o.jn[2] = a1.x;
        o.kn[0] = a1.y;
        o.kn[1] = a2.x;
        o.kn[2] = a2.y;
        o.r = a3.x;
        o.f[8] = a3.y;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const v2 t = *(const v2 *)(rb + 3072 + g * 256);
            o.f[2 * g] = t.x;
            o.f[2 * g + 1] = t.y;
        }
    } else if constexpr (NEQ == 3) {
        typedef float v4 __attribute__((ext_vector_type(4)));
        typedef float v3 __attribute__((ext_vector_type(3)));
        const v4 a = *(const v4 *)b;
        const v3 k = *(const v3 *)(b + 768);
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            o.jn[n] = a[n];
            o.kn[n] = k[n];
        }
        o.r = a[3];
    } else {
        typedef double v2 __attribute__((ext_vector_type(2)));
        const v2 a = *(const v2 *)b, c = *(const v2 *)(b + 1024);
        o.jn[0] = a.x;
        o.kn[0] = a.y;
        o.r = c.x;
        o.f[0] = c.y;
    }
    if constexpr (NEQ == 3 && sizeof(T) == 8) {
        // no wider than the three words: a register loaded for nothing is reused at once, and
        // writing it would wait for every LDS read in flight
        typedef double v2 __attribute__((ext_vector_type(2)));
        const v2 t = *(const v2 *)e;
        o.e[0] = t.x;
        o.e[1] = t.y;
        o.e[2] = e[2];
    } else {
        o.e[0] = e[0];
    }
}

// One step of ilusol3 / ilusol1 at this lane's row: the forward part (ref/ilusol.f:127-202 and
// 502-540: the j-term, then the k-term) or the backward part (ref/ilusol.f:353-469 and
// 560-591: the k-term, then the j-term).  own: the row's result of the step before (in) and
// of this one (out).  T = double: the reference's arithmetic; float: the scaled form.
// first part: the sum of this lane's equation (v: that equation of `own`)
template <int NEQ, bool FWD, typename T>
SMAC_DEV T band_sum(const Ops<NEQ, T> &o, const T own[NEQ], T v)
{
    T t = o.r;
    if constexpr (NEQ == 3 && sizeof(T) == 4) {
        // t += -b x.  A lane keeps its own equation only: the fused multiply-adds take the three
        // equations' values from the quad, of the row's last result (v) and of the row before
        // (x, which is the quad before's v, or e).  A DPP operand is read no sooner than two
        // instructions after it was written.
        T x = o.e[0];
        if constexpr (FWD)
            asm("s_nop 1\n\t"
                "v_mov_b32_dpp %1, %2 row_shr:4 row_mask:0xf bank_mask:0xe\n\t"
                "v_fmac_f32_dpp %0, %2, -%3 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
                "v_fmac_f32_dpp %0, %2, -%4 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
                "v_fmac_f32_dpp %0, %2, -%5 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf\n\t"
                "v_fmac_f32_dpp %0, %1, -%6 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
                "v_fmac_f32_dpp %0, %1, -%7 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
                "v_fmac_f32_dpp %0, %1, -%8 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf"
                : "+&v"(t), "+&v"(x)
                : "v"(v), "v"(o.jn[0]), "v"(o.jn[1]), "v"(o.jn[2]), "v"(o.kn[0]), "v"(o.kn[1]),
                  "v"(o.kn[2]));
        else
            asm("s_nop 1\n\t"
                "v_mov_b32_dpp %1, %2 row_shr:4 row_mask:0xf bank_mask:0xe\n\t"
                "s_nop 1\n\t"
                "v_fmac_f32_dpp %0, %1, -%6 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
                "v_fmac_f32_dpp %0, %1, -%7 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
                "v_fmac_f32_dpp %0, %1, -%8 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf\n\t"
                "v_fmac_f32_dpp %0, %2, -%3 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
                "v_fmac_f32_dpp %0, %2, -%4 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
                "v_fmac_f32_dpp %0, %2, -%5 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf"
                : "+&v"(t), "+&v"(x)
                : "v"(v), "v"(o.jn[0]), "v"(o.jn[1]), "v"(o.jn[2]), "v"(o.kn[0]), "v"(o.kn[1]),
                  "v"(o.kn[2]));
    } else {
        T nb[NEQ];
#pragma unroll
        for (int n = 0; n < NEQ; ++n) nb[n] = from_row_before<NEQ>(own[n], o.e[n]);
        auto part = [&](const T *b, const T *x) {
#pragma unroll
            for (int n = 0; n < NEQ; ++n) t = t - b[n] * x[n];
        };
        if constexpr (FWD) {
            part(o.jn, own);
            part(o.kn, nb);
        } else {
            part(o.kn, nb);
            part(o.jn, own);
        }
    }
    return t;
}
// second part: the row's result from the equations' sums, t that of this lane's; returns this
// lane's equation of it (c0, c1: whether that is the first, the second)
template <int NEQ, typename T>
SMAC_DEV T band_solve(const Ops<NEQ, T> &o, T t, T own[NEQ], bool c0, bool c1)
{
    if constexpr (NEQ == 3 && sizeof(T) == 8) {
        lu_solve3<double>(o.f, quad_lane<0>(t), quad_lane<1>(t), quad_lane<2>(t), own);
        // kept as selects (not sunk into branches)
        const T v = keep(c1 ? own[1] : own[2]);
        return keep(c0 ? own[0] : v);
    } else if constexpr (NEQ == 3) {
        // scaled form: the blocks and the rhs already carry the inverse diagonal
        return t;
    } else {
        return own[0] = o.f[0] * t;
    }
}

// f(0), f(1), .. with constant arguments, until one returns false
template <class Fn, int... U>
static __device__ __forceinline__ bool ring_round(Fn &f, std::integer_sequence<int, U...>)
{
    return (f(std::integral_constant<int, U>{}) && ...);
}

// One band of one case: blk is the band's place in dispatch order (forward bands bottom up,
// backward bands top down, so that every band is dispatched after the band it waits for).
template <int NEQ, bool FWD, typename T, class F = Form<NEQ, T>>
SMAC_DEV void band_run(const Dims &d, const LusgsWs &w, int blk)
{
    static_assert(F::RING % F::SUB == 0 && F::RING % LOADERS == 0 && F::RING % (F::AHEAD + 1) == 0 &&
                      F::RING - F::FLY * LOADERS > 2 * F::SUB,
                  "ring");
    constexpr int NDMA = (F::IMG + 1023) / 1024;
    static_assert(F::FLY * NDMA <= 63, "vmcnt budget");
    static_assert(F::SUB + F::AHEAD + 3 * F::SKEW <= OVER<F> && OVER<F> <= HP0,
                  "the sweeps run past their ends within the padding");
    __shared__ BandLds<F, T> L;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nband = w.nband;
    const int b = FWD ? blk : nband - 1 - blk;
    const int k0 = b * w.rows;
    const int klast = (k0 + w.rows < d.km ? k0 + w.rows : d.km) - 1;
    const int nrow = klast - k0 + 1;
    const int dir = FWD ? 1 : -1;
    const int h0 = FWD ? k0 : d.jm - 1 + klast;
    const int nsteps = d.jm - 1 + nrow + (nrow - 1) / 4 * F::SKEW;
    auto behind = [&](int q) { return q / 4 * F::SKEW; };   // steps that row slot q runs behind
    constexpr int SUB = F::SUB;
    const int nexec = (nsteps + SUB - 1) / SUB * SUB, nload = nexec + F::AHEAD;
    // row slot q of the band, in sweep order: the row that takes the hand-over is slot 0; slots
    // without a row work on the padding row ks - 1
    auto row_of = [&](int q) { return q < nrow ? (FWD ? k0 + q : klast - q) : w.ks - 1; };
    const int kin = FWD ? k0 : klast, kout = FWD ? klast : k0;
    const bool has_in = FWD ? b > 0 : b + 1 < nband, has_out = FWD ? b + 1 < nband : b > 0;
    const long fpitch = (long)(w.ks / F::ROWS) * F::FB * dir, bpitch = (long)(w.ks / F::ROWS) * F::BB * dir;
    // edge regions: forward sweep bands 0..nband-1, backward sweep nband..2*nband-1
    unsigned long long *ebase = w.edge + (FWD ? 0 : (long)nband * w.epitch);

    for (int i = threadIdx.x; i < F::RING * F::EDGE; i += BAND_LANES * BAND_WAVES)
        L.edge[i / F::EDGE][i % F::EDGE] = (T)0;
    if (threadIdx.x < 4) L.cnt[threadIdx.x] = threadIdx.x == LOADERS && !has_in ? 0x7fffffff : 0;
    if (threadIdx.x == 4) L.consumed = 0;
    __syncthreads();

    if (wave <= LOADERS && wave > 0) {
        // ---- loader: this lane's 16 bytes of each DMA instruction, from the chunk that holds
        // its row (a band may cover rows of two chunks, and the backward order is reversed)
        const char *src[NDMA];
        long pitch[NDMA];
#pragma unroll
        for (int i = 0; i < NDMA; ++i) {
            const int o = i * 1024 + lane * 16;
            int q, off;                 // row slot; offset of the piece in the chunk of row 0
            if constexpr (NEQ == 3) {
                const int lp = sizeof(T) == 8 ? 3072 : 1536;
                q = o < lp ? o % 768 / 48 : (o - lp) % 256 / 16;
                off = o < lp ? o / 768 * 768 + o % 48 : lp + (o - lp) / 256 * 256;
            } else {
                q = o % 1024 / 16;
                off = o / 1024 * 1024;
            }
            const int k = row_of(q), tile = k / F::ROWS, kt = k % F::ROWS;
            off += kt * (NEQ == 3 && o < (sizeof(T) == 8 ? 3072 : 1536) ? 48 : 16);
            const bool own = FWD || o >= F::BOWN;
            src[i] = (own ? fwd_chunk<F>(w, h0, tile) : bwd_chunk<F>(w, h0, tile)) + off;
            pitch[i] = own ? fpitch : bpitch;
            src[i] -= behind(q) * pitch[i];
        }
        const int first = wave - 1;
        const unsigned landed = lds_addr(&L.cnt[first]), consumed = lds_addr(&L.consumed);
        int prog = 0, slot = first * F::IMG;
#pragma unroll
        for (int i = 0; i < NDMA; ++i) {
            src[i] += first * pitch[i];
            pitch[i] *= LOADERS;
        }
        for (int st = first; st < nload; st += LOADERS) {
            while (st >= prog + F::RING) {
                prog = cnt_ld_dma(consumed);
                if (st >= prog + F::RING) __builtin_amdgcn_s_sleep(1);
            }
#pragma unroll
            for (int i = 0; i < NDMA; ++i) {
                if ((i + 1) * 1024 <= F::IMG || lane * 16 < F::IMG - i * 1024)
                    dma16(src[i], L.ring + slot + i * 1024);
                src[i] += pitch[i];
            }
            slot += LOADERS * F::IMG;
            if (slot >= F::RING * F::IMG) slot -= F::RING * F::IMG;
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(F::FLY * NDMA));
            // this wave's steps before the FLY latest ones have landed
            cnt_st_dma(landed, st - (F::FLY - 1) * LOADERS);
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        // no more to wait for
        cnt_st_dma(landed, 0x7fffffff);
        return;
    }
    if (wave == LOADERS + 1) {
        // ---- hand-over: the words of BS steps per poll, one word per lane; the prefix of them
        // that has been written goes to LDS.  One poll at a time: with four in flight a slot is
        // seen sooner, but the waves' polls (each up to 63 words in as many sectors, past the
        // caches) hold up one another and the operands: 945x241 alone FP64 558 us a pass instead
        // of 548, a batch of 64 cases 5.16 ms instead of 5.10, FP32-LHS 3.39 instead of 3.36.
        if (!has_in) return;
        constexpr int BS = F::RING < 21 ? F::RING : (NEQ == 3 ? 21 : F::RING);
        const int i = lane / NEQ, word = lane % NEQ;
        // the slot of column j = h - kin
        const unsigned long long *p0 = ebase + (long)(b - dir) * w.epitch +
                                       (long)(h0 - kin + EPAD) * 4 + word;
        int base = 0, lim = F::RING, spin = 0;
        bool broken = false;
        while (base < nload) {
            const int st = base + i;
            const unsigned long long v = __hip_atomic_load(
                p0 + (long)dir * (st < nload ? st : nload - 1) * 4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (base + BS > lim) lim = cnt_ld(&L.consumed) + F::RING;
            const int top = base + BS < lim ? base + BS : lim;
            const int end = top < nload ? top : nload;    // steps this poll may hand over
            const bool none = edge_empty(v) && !broken;
            const unsigned long long missing = __builtin_amdgcn_ballot_w64(none && i < BS && st < end);
            const int upto = missing ? base + __builtin_ctzll(missing) / NEQ : end;
            if (upto > base) {
                if (i < BS && st < upto) {
                    T x;
                    slot_value(edge_empty(v) ? 0ull : v, x);
                    L.edge[st % F::RING][word] = x;
                }
                asm volatile("" ::: "memory");
                base = upto;
                if (lane == 0) cnt_st(&L.cnt[LOADERS], base < nload ? base : 0x7fffffff);
                spin = 0;
            } else if (base < lim && ++spin > EDGE_SPIN_MAX) {
                broken = true;
                if (lane == 0) atomicOr(w.stall, 1);
            }
        }
        return;
    }
    // ---- the computing wavefront
    __builtin_amdgcn_s_setprio(3);
    const int c = NEQ == 3 ? ((lane & 3) < 2 ? lane & 3 : 2) : 0, q = NEQ == 3 ? lane >> 2 : lane;
    const bool c0 = c == 0, c1 = c == 1;
    const int krow = row_of(q), ktile = krow / F::ROWS, kk = krow % F::ROWS;
    const unsigned char *lb = L.ring + (NEQ == 3 ? q * 48 + c * 16 : q * 16), *rb = L.ring + q * 16;
    constexpr bool YB = FWD && F::Y_BWD;
    char *out = r_of<F>(YB ? bwd_chunk<F>(w, h0, ktile) : fwd_chunk<F>(w, h0, ktile), kk, c);
    const long opitch = YB ? bpitch : fpitch;
    out -= behind(q) * opitch;
    const rsrc_t rE = mk_rsrc(ebase + (long)b * w.epitch, (unsigned)w.epitch * 8u);
    const unsigned eo = has_out && q == nrow - 1 ? 8u * c : 0x80000000u;
    unsigned es = (unsigned)(h0 - dir * behind(nrow - 1) - kout + EPAD) * 32u;

    // the least of the four counters (three loaders, the hand-over), in every lane
    static_assert(LOADERS == 3, "four counters in one read");
    typedef int v4i __attribute__((ext_vector_type(4)));
    auto counts = [&]() -> v4i { return *(const v4i *)L.cnt; };
    auto least = [](v4i a) {
        const int x = a.x < a.y ? a.x : a.y, y = a.z < a.w ? a.z : a.w;
        return x < y ? x : y;
    };
    auto reached = [](int v, int n) { return __builtin_amdgcn_ballot_w64(v < n) == 0; };
    auto await = [&](int n) {
        while (!reached(least(counts()), n)) asm volatile("" ::: "memory");   // read again
        asm volatile("" ::: "memory");
    };
    T own[NEQ];
#pragma unroll
    for (int n = 0; n < NEQ; ++n) own[n] = (T)0;
    T v = (T)0;                   // this lane's equation of the row's last result
    // skewed rows: a step's hand-over values of row slots 0, 4, 8 and 12, four words each; the
    // lanes of slots 3, 7 and 11 pass theirs on, the others write a word that is not read
    const int take = F::SKEW > 0 ? lane / 16 * 4 + c : 0;
    const int pass = lane < 48 && lane % 16 >= 12 ? lane / 16 * 4 + 4 + lane % 4 : 16 + lane % 4;
    constexpr int A = F::AHEAD;
    Ops<NEQ, T> s[A + 1];
    await(A);
#pragma unroll
    for (int u = 0; u < A; ++u)
        read_ops<NEQ, T>(s[u], lb + u * F::IMG, rb + u * F::IMG, L.edge[u] + take);
    v4i last = {0, 0, 0, 0};
    int st = 0;
    // the step in ring slot u; false once the band is done (looked at every SUB steps)
    auto one = [&](auto uc) -> bool {
        constexpr int u = decltype(uc)::value, R = F::RING;
        if constexpr (u % SUB == 0) {
            if (st >= nexec) return false;
            // the counters as read SUB / 2 steps ago usually suffice
            cnt_st(&L.consumed, st);     // the slots of the steps before st are free
            if (__builtin_expect(!reached(least(last), st + SUB + A), 0)) await(st + SUB + A);
            asm volatile("" ::: "memory");
            st += SUB;
        }
        if constexpr (u % SUB == SUB / 2) last = counts();
        constexpr int un = (u + A) % R;
        read_ops<NEQ, T>(s[un % (A + 1)], lb + un * F::IMG, rb + un * F::IMG, L.edge[un] + take);
        const T t = band_sum<NEQ, FWD, T>(s[u % (A + 1)], own, v);
        v = band_solve<NEQ, T>(s[u % (A + 1)], t, own, c0, c1);
        // to the four rows that run SKEW steps behind: they read it in the next step, for the
        // step AHEAD of that
        if constexpr (F::SKEW > 0) L.edge[(u + A + 1) % R][pass] = v;
        *(T *)out = v;                       // slots without a row: padding
        out += opitch;
        unsigned lo, hi;
        slot_word(v, lo, hi);
        edge_st(lo, hi, rE, eo, es);
        es += 32u * dir;
        __builtin_amdgcn_sched_barrier(0);
        return true;
    };
    while (ring_round(one, std::make_integer_sequence<int, F::RING>{})) {}
}

template <int NEQ, bool FWD, typename T, class F>
__global__ void __launch_bounds__(BAND_LANES * BAND_WAVES)
k_band(Dims d, LusgsWs w)
{
    band_run<NEQ, FWD, T, F>(d, w, (int)blockIdx.x);
}

// The bands of several cases in one launch: workgroup i runs band map[i].y of case map[i].x.
// The map lists each case's bands contiguously in dispatch order, so every wait is on a
// workgroup dispatched earlier.
// a workspace out of a table in memory
SMAC_DEV LusgsWs ws_global(const LusgsWs &t)
{
    LusgsWs w = t;
    w.lhs = as_global(t.lhs);
    w.edge = as_global(t.edge);
    w.stall = as_global(t.stall);
    return w;
}

template <int NEQ, bool FWD, typename T, class F>
__global__ void __launch_bounds__(BAND_LANES * BAND_WAVES)
k_band_multi(const BandJob *__restrict__ jobs, const int2 *__restrict__ map,
             const int *__restrict__ active)
{
    const int2 m = map[blockIdx.x];
    // a stopped case: all of its bands leave, so none waits on another
    if (active && active[jobs[m.x].bcase] == 0) return;
    const Dims d = jobs[m.x].d;
    const LusgsWs w = ws_global(jobs[m.x].w);
    band_run<NEQ, FWD, T, F>(d, w, m.y);
}

// ------------------------------------------------------------------------------------------

void lusgs_ws_shape(int jm, int km, int rows, int neqs, LusgsWs &w)
{
    const int most = neqs == 3 ? Form<3, double>::ROWS : Form<1, double>::ROWS;
    static_assert(Form<3, double>::ROWS == Form<3, float>::ROWS, "one shape for both precisions");
    w.rows = rows < 1 ? 1 : (rows > most ? most : rows);
    w.nband = (km + w.rows - 1) / w.rows;
    // row ks-1 is padding (row slots without a row work there)
    w.ks = (km + 1 + most - 1) / most * most;
    w.H = jm + km - 2;
    w.epitch = (jm + 2 * EPAD) * 4;
    w.nedge = 2L * w.nband * w.epitch;
}

// sizes for the FP64 system (the FP32-LHS one needs less and fits the same allocation)
long lusgs_ws_lhs_bytes(const LusgsWs &w, int neqs)
{
    using F3 = Form<3, double>;
    using F1 = Form<1, double>;
    static_assert(Form<3, float>::FB + Form<3, float>::BB <= F3::FB + F3::BB, "FP32 fits");
    const long pos = (long)(w.H + 1 + 2 * HP0) * w.ks;
    return neqs == 3 ? pos / F3::ROWS * (F3::FB + F3::BB) : pos / F1::ROWS * (F1::FB + F1::BB);
}

template <typename LT, int NEQ>
void lusgs_pre(hipStream_t sm, const Dims &d, const LusgsWs &w, const double *rhs, const LT *btc,
               const LT *bjm, const LT *bjp, const LT *bkm, const LT *bkp, LT *fac)
{
    hipLaunchKernelGGL((k_shear<LT, NEQ>), (shear_grid<LT, NEQ>(d, w)), dim3(TILE_THREADS), 0, sm,
                       d, w, rhs, btc, bjm, bkm, bjp, bkp, fac);
}

// The form of a launch of nblk bands beside which a launch of `beside` bands of the other system
// may run (launch gets it, and LDS to ask for beyond the kernel's own).
//
// A band waits for the band before it, which its launch dispatched earlier.  That one makes its way
// as long as the bands of the other launch, which wait for one another too, do not hold every place
// it could take.  As long as lusgs_bands_fit none does.  Beyond that the scalar system's bands take
// a ring small enough, and the mean flow's one large enough (FormMost asks for more LDS than it
// uses), that the units which hold all the mean-flow bands they can have room (and registers) for
// one of the scalar system's: those end then, and with them what holds up the others.  In the other
// forms a unit with a scalar band has no room for an FP64 one, and one full of FP32 bands none for a
// scalar one.
//
// A pass, in the forms of a single case and in these: 26 cases FP64 (276 + 69 bands) 2270 and 2290
// us, 64 cases (632 + 158) 5089 and 5095; FP32-LHS 16 of 945x241 (256 + 64) 1722 and 1696, 32 of
// them (512 + 128) 3301 and 3298, 32 cases (340 + 85) 1958 and 1973, 64 cases 3344 (the shortest
// ring, four bands a unit) and 3334; below, 12 cases (124 + 31) 825 and 856.  Alone, FP32 past two
// bands a unit takes the shortest ring: 64 cases without the SA 2580 and 2541 us.  (One row per lane in 64-row bands, of which the 64 cases
// had 158, took 0.32 ms for a forward sweep of theirs beside the SA, and 3.54 for a pass.  It takes
// 0.48 now: on a chip full of bands the sixteen-row ones lose their gain to hand-overs.)
constexpr int LDS_UNIT = 160 * 1024, LDS_GRAIN = 1280;
constexpr int lds_grains(int bytes) { return (bytes + LDS_GRAIN - 1) / LDS_GRAIN * LDS_GRAIN; }
template <class F, typename T> constexpr int lds_of(int room = 0)
{
    return lds_grains((int)sizeof(BandLds<F, T>) + room);
}
constexpr int MOST_ROOM = LDS_UNIT / 4 + 16 - (int)sizeof(BandLds<FormMost, float>);
constexpr bool leaves_room(int mean)
{
    return LDS_UNIT % mean >= lds_of<FormMany<1, double>, double>();
}
static_assert(leaves_room(lds_of<Form<3, double>, double>()), "FP64");
static_assert(leaves_room(lds_of<FormMany<3, float>, float>()), "FP32");
static_assert(leaves_room(lds_of<FormMost, float>(MOST_ROOM)), "FP32, many");

template <typename LT, int NEQ, class Launch>
static void band_form(int nblk, int beside, Launch launch)
{
    const bool crowd = beside > 0 && !lusgs_bands_fit(nblk + beside);
    if constexpr (NEQ == 3 && sizeof(LT) == 4) {
        if (nblk > 2 * LUSGS_UNITS) return launch(FormMost{}, crowd ? MOST_ROOM : 0);
    }
    if constexpr (NEQ == 1 || sizeof(LT) == 4) {
        if (crowd) return launch(FormMany<NEQ, LT>{}, 0);
    }
    launch(Form<NEQ, LT>{}, 0);
}

template <typename LT, int NEQ>
void lusgs_band(hipStream_t sm, const Dims &d, const LusgsWs &w, bool fwd)
{
    const dim3 blk(BAND_LANES * BAND_WAVES);
    band_form<LT, NEQ>(w.nband, w.beside, [&](auto form, int room) {
        using F = decltype(form);
        if (fwd)
            hipLaunchKernelGGL((k_band<NEQ, true, LT, F>), dim3(w.nband), blk, room, sm, d, w);
        else
            hipLaunchKernelGGL((k_band<NEQ, false, LT, F>), dim3(w.nband), blk, room, sm, d, w);
    });
}

template <typename LT, int NEQ>
void lusgs_band_multi(hipStream_t sm, const BandJob *jobs, const int2 *map, int nblk, int beside,
                      bool fwd, const int *active)
{
    if (nblk <= 0) return;
    const dim3 blk(BAND_LANES * BAND_WAVES);
    band_form<LT, NEQ>(nblk, beside, [&](auto form, int room) {
        using F = decltype(form);
        if (fwd)
            hipLaunchKernelGGL((k_band_multi<NEQ, true, LT, F>), dim3(nblk), blk, room, sm, jobs, map, active);
        else
            hipLaunchKernelGGL((k_band_multi<NEQ, false, LT, F>), dim3(nblk), blk, room, sm, jobs, map, active);
    });
}

template <typename LT, int NEQ>
void lusgs_mid(hipStream_t sm, const Dims &d, const LusgsWs &w)
{
    if (NEQ == 3 && sizeof(LT) == 4) return;   // scaled form: D^-1 (D y) = y
    hipLaunchKernelGGL((k_mid<LT, NEQ>), dim3(mid_blocks<NEQ>(w)), dim3(256), 0, sm, d, w);
}

template <typename LT, int NEQ>
void lusgs_post(hipStream_t sm, const Dims &d, const LusgsWs &w, const WakePairs &wk,
                const double *q, double *dq, double *rhs)
{
    hipLaunchKernelGGL((k_unshear<NEQ, LT>), unshear_grid(d, w), dim3(TILE_THREADS), 0, sm, d, w,
                       false, dq, WakeIn{wk, q, rhs});
}

// ---- multi-case launches ------------------------------------------------------------------

template <typename LT, int NEQ>
ShearArgs shear_args(const Dims &d, const LusgsWs &w, const double *rhs, const LT *btc,
                     const LT *bjm, const LT *bjp, const LT *bkm, const LT *bkp, LT *fac)
{
    const dim3 g = shear_grid<LT, NEQ>(d, w);
    return ShearArgs{g.x, g.y, d, w, rhs, btc, bjm, bkm, bjp, bkp, fac};
}

template <typename LT, int NEQ>
MidArgs mid_args(const Dims &d, const LusgsWs &w)
{
    if (NEQ == 3 && sizeof(LT) == 4) return MidArgs{0u, 1u, d, w};   // scaled form
    return MidArgs{mid_blocks<NEQ>(w), 1u, d, w};
}

UnshearArgs unshear_args(const Dims &d, const LusgsWs &w, double *dst)
{
    const dim3 g = unshear_grid(d, w);
    return UnshearArgs{g.x, g.y, d, w, dst};
}

template <typename LT, int NEQ>
struct CShear {
    using Args = ShearArgs;
    static constexpr int THREADS = TILE_THREADS;
    static SMAC_DEV void run(const Blk &b, const Args &a)
    {
        b_shear<LT, NEQ>(b, a.d, ws_global(a.w), as_global(a.rhs), (const LT *)as_global(a.btc),
                         (const LT *)as_global(a.bjm), (const LT *)as_global(a.bkm),
                         (const LT *)as_global(a.bjp), (const LT *)as_global(a.bkp),
                         a.fac ? (LT *)as_global(a.fac) : nullptr);
    }
};
template <typename LT, int NEQ>
struct CMid {
    using Args = MidArgs;
    static constexpr int THREADS = 256;
    static SMAC_DEV void run(const Blk &b, const Args &a) { b_mid<LT, NEQ>(b, a.d, ws_global(a.w)); }
};
template <typename LT, int NEQ>
struct CUnshear {
    using Args = UnshearArgs;
    static constexpr int THREADS = TILE_THREADS;
    static SMAC_DEV void run(const Blk &b, const Args &a)
    {
        b_unshear<NEQ, LT>(b, a.d, ws_global(a.w), false, as_global(a.dst), WakeIn{});
    }
};

template <class C>
static void multi_launch(hipStream_t sm, const MultiTab<typename C::Args> &t)
{
    if (t.n > 0 && t.nblk > 0)
        hipLaunchKernelGGL(k_multi<C>, dim3(t.nblk), dim3(C::THREADS), 0, sm, t.args, t.start, t.n,
                           t.item_case, t.active);
}

template <typename LT, int NEQ> void multi_shear(hipStream_t sm, const MultiTab<ShearArgs> &t)
{
    multi_launch<CShear<LT, NEQ>>(sm, t);
}
template <typename LT, int NEQ> void multi_mid(hipStream_t sm, const MultiTab<MidArgs> &t)
{
    multi_launch<CMid<LT, NEQ>>(sm, t);
}
template <typename LT, int NEQ> void multi_unshear(hipStream_t sm, const MultiTab<UnshearArgs> &t)
{
    multi_launch<CUnshear<LT, NEQ>>(sm, t);
}

template ShearArgs shear_args<double, 1>(const Dims &, const LusgsWs &, const double *,
                                         const double *, const double *, const double *,
                                         const double *, const double *, double *);
template ShearArgs shear_args<double, 3>(const Dims &, const LusgsWs &, const double *,
                                         const double *, const double *, const double *,
                                         const double *, const double *, double *);
template ShearArgs shear_args<float, 3>(const Dims &, const LusgsWs &, const double *,
                                        const float *, const float *, const float *,
                                        const float *, const float *, float *);
template MidArgs mid_args<double, 1>(const Dims &, const LusgsWs &);
template MidArgs mid_args<double, 3>(const Dims &, const LusgsWs &);
template MidArgs mid_args<float, 3>(const Dims &, const LusgsWs &);
template void multi_shear<double, 1>(hipStream_t, const MultiTab<ShearArgs> &);
template void multi_shear<double, 3>(hipStream_t, const MultiTab<ShearArgs> &);
template void multi_shear<float, 3>(hipStream_t, const MultiTab<ShearArgs> &);
template void multi_mid<double, 1>(hipStream_t, const MultiTab<MidArgs> &);
template void multi_mid<double, 3>(hipStream_t, const MultiTab<MidArgs> &);
template void multi_mid<float, 3>(hipStream_t, const MultiTab<MidArgs> &);
template void multi_unshear<double, 1>(hipStream_t, const MultiTab<UnshearArgs> &);
template void multi_unshear<double, 3>(hipStream_t, const MultiTab<UnshearArgs> &);
template void multi_unshear<float, 3>(hipStream_t, const MultiTab<UnshearArgs> &);

template <typename LT, int NEQ>
static void launch_lusgs(hipStream_t sm, const Dims &d, const LusgsWs &w, const WakePairs &wk,
                         const double *q, double *dq, double *rhs, const LT *btc, const LT *bjm,
                         const LT *bjp, const LT *bkm, const LT *bkp, LT *fac, bool rhs_out)
{
    lusgs_pre<LT, NEQ>(sm, d, w, rhs, btc, bjm, bjp, bkm, bkp, fac);
    if (w.ev_fwd[0]) (void)hipEventRecord(w.ev_fwd[0], sm);
    lusgs_band<LT, NEQ>(sm, d, w, true);
    if (w.ev_fwd[1]) (void)hipEventRecord(w.ev_fwd[1], sm);
    lusgs_mid<LT, NEQ>(sm, d, w);
    if (rhs_out)   // before the backward sweep writes dq in its place
        hipLaunchKernelGGL((k_unshear<NEQ, LT>), unshear_grid(d, w), dim3(TILE_THREADS), 0, sm, d, w,
                           true, rhs, WakeIn{});
    lusgs_band<LT, NEQ>(sm, d, w, false);
    lusgs_post<LT, NEQ>(sm, d, w, wk, q, dq, rhs);
}

template <typename LT>
void launch_lusgs3(hipStream_t sm, const Dims &d, const LusgsWs &w, const WakePairs &wk,
                   const double *q, double *dq, double *rhs, const LT *btc, const LT *bjm,
                   const LT *bjp, const LT *bkm, const LT *bkp, LT *fac, bool rhs_out)
{
    launch_lusgs<LT, 3>(sm, d, w, wk, q, dq, rhs, btc, bjm, bjp, bkm, bkp, fac, rhs_out);
}

void launch_lusgs1(hipStream_t sm, const Dims &d, const LusgsWs &w, const WakePairs &wk,
                   const double *q, double *dq, double *rhs, const double *btc, const double *bjm,
                   const double *bjp, const double *bkm, const double *bkp, double *fac,
                   bool rhs_out)
{
    launch_lusgs<double, 1>(sm, d, w, wk, q, dq, rhs, btc, bjm, bjp, bkm, bkp, fac, rhs_out);
}

#define PHASES(LT, NEQ)                                                                        \
    template void lusgs_pre<LT, NEQ>(hipStream_t, const Dims &, const LusgsWs &, const double *, \
                                     const LT *, const LT *, const LT *, const LT *, const LT *, \
                                     LT *);                                                    \
    template void lusgs_band<LT, NEQ>(hipStream_t, const Dims &, const LusgsWs &, bool);       \
    template void lusgs_band_multi<LT, NEQ>(hipStream_t, const BandJob *, const int2 *, int,   \
                                            int, bool, const int *);                                \
    template void lusgs_mid<LT, NEQ>(hipStream_t, const Dims &, const LusgsWs &);              \
    template void lusgs_post<LT, NEQ>(hipStream_t, const Dims &, const LusgsWs &,              \
                                      const WakePairs &, const double *, double *, double *);
PHASES(double, 3)
PHASES(float, 3)
PHASES(double, 1)
#undef PHASES

template void launch_lusgs3<double>(hipStream_t, const Dims &, const LusgsWs &, const WakePairs &,
                                    const double *, double *, double *, const double *,
                                    const double *, const double *, const double *,
                                    const double *, double *, bool);
template void launch_lusgs3<float>(hipStream_t, const Dims &, const LusgsWs &, const WakePairs &,
                                   const double *, double *, double *, const float *,
                                   const float *, const float *, const float *, const float *,
                                   float *, bool);

}  // namespace smac
