/*
 * hd_thomas.h -- the speculative parallel Thomas solve shared by the ADI and
 * FS run kernels (one wave of 64 lanes per tridiagonal system, rows in LDS).
 */
#ifndef HD_THOMAS_H
#define HD_THOMAS_H

#include <hip/hip_runtime.h>

#include "hd_fastdiv.h"

namespace hd_spec {

constexpr int kSpecWave = 64;

/* ------------------------------------------- speculative parallel Thomas
 *
 * The forward elimination of tridiag (UVZSolver_multithread.cu:203-228),
 *   e_i = A_i ap_{i-1} + B_i,  ap_i = -C_i / e_i,  bp_i = (D_i - A_i bp_{i-1}) / e_i,
 * is a serial chain of a multiply, an add and a correctly rounded division per
 * row.  In exact arithmetic (ap, bp) = (p / q, r / q) where (p, q, r) follows
 * the linear recurrence v_i = M_i v_{i-1},
 *   M_i = [[0, -C_i, 0], [A_i, B_i, 0], [0, D_i, -A_i]],
 * so each lane composes the matrices of its own rows, an inclusive scan over
 * the wave (DPP row shifts and broadcasts) composes the prefixes, and every
 * lane obtains an estimate, good to
 * a few ulps, of the state after each earlier lane's rows.  The recurrence
 * contracts on these systems (each continuity / momentum pair reduces to a
 * diagonally dominant system in z), so two rounded trajectories that start a
 * few ulps apart become bit-identical after a few tens of rows.  A lane
 * therefore runs the exact recurrence -- the same IEEE operations in the same
 * order as the serial solve -- from the estimate of the state kSpecWF rows
 * before its own rows, through its own rows, and
 * the result is verified exactly: the state a lane had on entering its rows
 * must equal, bit for bit, the state its predecessor produced at its last
 * row.  Lane 0 starts from the exact state; by induction every lane that
 * passes is exact, and the first lane that fails is recomputed serially from
 * its verified predecessor, after which its successor is tested again.  The
 * result equals the serial solve's bits in every case; the speculation only
 * shortens the critical path from the run's length to about kSpecWF + L rows
 * (L = rows per lane).  Back substitution, x_i = bp_i + ap_i x_{i+1}, is an
 * affine chain and is treated the same way with 2-entry affine maps.
 *
 * What bounds it, and the layout.  One wave works alone on a run, so the time
 * is the length of its dependent chain: about 7 cycles per FP64 operation, 75
 * per division, 65 per LDS read that is waited for, 140 per row with two
 * divisions, and 50 more where a row sits behind its own branch
 * (microbenchmarks on this part).  Hence
 *  - the rows per lane L are a power of two, known to the compiler (one copy
 *    of the sweep for each), and row r sits at LDS position
 *    (r mod L) * S + r / L: the lanes of a step read consecutive words
 *    whatever L is, every row of the warm-up is at a fixed distance, and no
 *    row needs a branch: rows that a lane's warm-up would read outside the
 *    sweep are identity rows written there (16 before row 0, which hand on
 *    the entry state, and 32 identity factors after the last row for the
 *    back substitution);
 *  - a row takes one reciprocal for its two quotients (hd_fastdiv.h), with
 *    the division's own bits (95 cycles); where a value leaves the range in
 *    which that holds, the wave runs the sweep again with divisions;
 *  - matrices are normalised once per lane before the scan, not in it (64
 *    factors with entries at most 1 stay far inside the exponent range, and
 *    an estimate that does overflow only costs a repair).
 *
 * Repairs: while a flow starts from
 * rest, bp decays ahead of the waves as fast as the estimate's relative
 * error and never merges, so long stretches of lanes fail with their ap
 * already exact.  Then every row's divisor is known, and a failing lane
 * redoes only its bp chain, from registers, with known reciprocals. */
constexpr int kSpecWF = 16;           /* forward warm-up rows after the estimate */
constexpr int kSpecWB = 32;           /* back-substitution warm-up rows */
constexpr int kSpecMaxLg = 3;         /* rows per lane of one sweep: 1, 2, 4 or 8 */

/* words between the planes r mod L of an LDS array: the warm-up before row
 * 0, 64 lanes, the back substitution's warm-up after them */
constexpr int spec_stride(int lg) { return kSpecWave + ((kSpecWF + kSpecWB) >> lg); }
/* LDS position of row r (>= -kSpecWF) with 2^lg rows per lane */
struct SpecMap {
    int lg;
    __device__ __forceinline__ int pos(int r) const
    {
        return ((r + kSpecWF) & ((1 << lg) - 1)) * (kSpecWave + ((kSpecWF + kSpecWB) >> lg)) + ((r + kSpecWF) >> lg);
    }
};
/* words per LDS array of a sweep of at most n rows, and two more, at
 * spec_words(n) - 2 and - 1, for the caller's own use; a multiple of 64, so
 * that one instruction reads the same position of two arrays */
constexpr int spec_words(int n)
{
    int lg = 0;
    while ((kSpecWave << lg) < n) ++lg;
    return (((spec_stride(lg) << lg) + 2 + 63) / 64) * 64;
}
__device__ __forceinline__ SpecMap spec_map(int n, int minlg = 0)
{
    const int lg = n <= 64 ? 0 : (n <= 128 ? 1 : (n <= 256 ? 2 : 3));
    return SpecMap{lg < minlg ? minlg : lg};
}

struct Mx {
    double a, b, c, d, e, f, g; /* [[a b 0] [c d 0] [e f g]] */
};

/* M_i X for the row matrix M_i of (A, B, C, D) */
__device__ __forceinline__ Mx mx_row(double A, double B, double C, double D, const Mx& X)
{
    Mx R;
    R.a = -C * X.c;
    R.b = -C * X.d;
    R.c = fma(A, X.a, B * X.c);
    R.d = fma(A, X.b, B * X.d);
    R.e = fma(D, X.c, -A * X.e);
    R.f = fma(D, X.d, -A * X.f);
    R.g = -A * X.g;
    return R;
}

/* X Y */
__device__ __forceinline__ Mx mx_mul(const Mx& X, const Mx& Y)
{
    Mx R;
    R.a = fma(X.a, Y.a, X.b * Y.c);
    R.b = fma(X.a, Y.b, X.b * Y.d);
    R.c = fma(X.c, Y.a, X.d * Y.c);
    R.d = fma(X.c, Y.b, X.d * Y.d);
    R.e = fma(X.e, Y.a, fma(X.f, Y.c, X.g * Y.e));
    R.f = fma(X.e, Y.b, fma(X.f, Y.d, X.g * Y.f));
    R.g = X.g * Y.g;
    return R;
}

/* Scale by a power of two (exact) so the largest entry lies in [0.5, 1):
 * only ratios of the composed state matter.  A zero, infinite or NaN maximum
 * has exponent 0 here and leaves X as it is. */
__device__ __forceinline__ void mx_norm(Mx& X)
{
    const double m = fmax(fmax(fmax(fabs(X.a), fabs(X.b)), fmax(fabs(X.c), fabs(X.d))),
                          fmax(fmax(fabs(X.e), fabs(X.f)), fabs(X.g)));
    const int s = -__builtin_amdgcn_frexp_exp(m);
    X.a = __builtin_amdgcn_ldexp(X.a, s); X.b = __builtin_amdgcn_ldexp(X.b, s);
    X.c = __builtin_amdgcn_ldexp(X.c, s); X.d = __builtin_amdgcn_ldexp(X.d, s);
    X.e = __builtin_amdgcn_ldexp(X.e, s); X.f = __builtin_amdgcn_ldexp(X.f, s);
    X.g = __builtin_amdgcn_ldexp(X.g, s);
}

/* A 64-bit value moved across lanes by a DPP mode (shifts by one lane, row
 * shifts within rows of 16 lanes, row broadcasts to later rows): a lane the
 * mode gives no source, or whose row ROWMASK leaves out, gets `old`. */
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_f64(double old, double src)
{
    const long long o = __double_as_longlong(old), v = __double_as_longlong(src);
    const int lo = __builtin_amdgcn_update_dpp((int)o, (int)v, CTRL, ROWMASK, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(v >> 32), CTRL, ROWMASK, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
/* the same where lanes without a source may get anything */
template <int CTRL>
__device__ __forceinline__ double dpp_any(double src)
{
    const long long v = __double_as_longlong(src);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
/* the previous lane's value (lane 0 keeps its own) */
__device__ __forceinline__ double lane_before(double v) { return dpp_f64<0x138, 0xF>(v, v); }

/* One step of the wave's inclusive prefix scan of row matrices: X := X Y
 * with Y the matrix of the source lane, where there is one (`has`). */
template <int CTRL>
__device__ __forceinline__ void mx_scan_step(Mx& X, bool has)
{
    Mx Y;
    Y.a = dpp_any<CTRL>(X.a); Y.b = dpp_any<CTRL>(X.b); Y.c = dpp_any<CTRL>(X.c); Y.d = dpp_any<CTRL>(X.d);
    Y.e = dpp_any<CTRL>(X.e); Y.f = dpp_any<CTRL>(X.f); Y.g = dpp_any<CTRL>(X.g);
    if (has) X = mx_mul(X, Y);
}

/* The same for the affine maps x -> al x + be of back substitution: the
 * source lane's map is applied first. */
template <int CTRL>
__device__ __forceinline__ void aff_scan_step(double& al, double& be, bool has)
{
    const double a2 = dpp_any<CTRL>(al), b2 = dpp_any<CTRL>(be);
    if (has) {
        be = fma(al, b2, be);
        al = al * a2;
    }
}

/* v of lane `l` (wave-uniform l) through the scalar unit */
__device__ __forceinline__ double readlane_f64(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

__device__ __forceinline__ bool same_bits(double x, double y)
{
    return __double_as_longlong(x) == __double_as_longlong(y);
}

/* One exact forward row, in the operation order of tridiag. */
__device__ __forceinline__ void thomas_row(double A, double B, double C, double D, double& ap, double& bp)
{
    const double e = A * ap + B;
    const double nap = -C / e;
    const double nbp = (D - (A * bp)) / e;
    ap = nap;
    bp = nbp;
}

/* bp of a row whose divisor e and refined reciprocal y are known: the
 * numerator is scaled up and the quotient down again (both exact while the
 * quotient is a normal number or zero), so that a bp that decays towards
 * the end of the exponent range stays in reach of the reciprocal form. */
__device__ __forceinline__ double bp_known_e(double A, double D, double bp, double e, double y, hd_div::Range& rg)
{
    const double q = hd_div::quot((D - (A * bp)) * 0x1p300, e, y);
    rg.num(q);
    return q * 0x1p-300;
}

/* A warm-up row: the same bits in all but extreme cases (whatever it
 * returns is verified before it counts). */
__device__ __forceinline__ void thomas_row_warm(double A, double B, double C, double D, double& ap, double& bp)
{
    const double e = A * ap + B;
    const double y = hd_div::rcp_refined(e);
    ap = hd_div::quot(C, -e, -y);
    bp = hd_div::quot(D - (A * bp), e, y);
}

/* The row of thomas_row with one reciprocal for both quotients: its bits
 * while rows_ok holds of `rg` and of the results (hd_fastdiv.h), if C and D
 * are not -0 (then neither numerator is) and C is in range. */
__device__ __forceinline__ void thomas_row_rcp(double A, double B, double C, double D, double& ap, double& bp,
                                               hd_div::Range& rg)
{
    const double e = A * ap + B;
    const double y = hd_div::rcp_refined(e);
    rg.den(e);
    ap = hd_div::quot(C, -e, -y);
    bp = bp_known_e(A, D, bp, e, y, rg);
}

/* whether the scaled quotients stood for normal numbers or zeros */
__device__ __forceinline__ bool rows_ok(const hd_div::Range& rg, double ap, double bp)
{
    return rg.den_ok() && rg.lo >= -720 && hd_div::finite(ap) && hd_div::finite(bp);
}

template <int LG>
__device__ __forceinline__ void spec_forward_lg(double* sA, double* sB, double* sC, double* sD, int n, double& ap,
                                                double& bp, int* fails)
{
    constexpr int L = 1 << LG, S = spec_stride(LG), m = kSpecWF >> LG; /* m: lanes of warm-up */
    constexpr SpecMap sm{LG};
    const int lane = threadIdx.x;
    const int kl = (n - 1) >> LG;       /* the last lane with rows */
    const bool act = lane <= kl;
    const int own = lane + m;           /* position of the lane's first row */
    /* rows -16 .. -1 hand on the entry state, rows after n - 1 fill the last lane */
    if (lane < kSpecWF) {
        const int p = sm.pos(lane - kSpecWF);
        sA[p] = 0.0; sB[p] = 1.0; sC[p] = -ap; sD[p] = bp;
    } else {
        const int r = n + lane - kSpecWF;
        if (r < ((kl + 1) << LG)) {
            const int p = sm.pos(r);
            sA[p] = 0.0; sB[p] = 1.0; sC[p] = 0.0; sD[p] = 0.0;
        }
    }
    __syncthreads();
    /* the lane's own rows, composed, and what the reciprocal form asks of C and D */
    double A[L], B[L], C[L], D[L];
    bool nz = false;
    hd_div::Range rc;
#pragma unroll
    for (int q = 0; q < L; ++q) {
        const int p = q * S + own;
        A[q] = sA[p]; B[q] = sB[p]; C[q] = sC[p]; D[q] = sD[p];
    }
#pragma unroll
    for (int q = 0; q < L; ++q) {
        nz = nz || hd_div::neg_zero(C[q]) || hd_div::neg_zero(D[q]);
        rc.num(C[q]);
    }
    const bool cd = !nz && rc.lo >= -900;
    bool plain = __any(act && !cd);
    const bool exact = lane <= m;       /* starts from the entry state */
    double a0 = ap, b0 = bp;
    if (n > kSpecWF + L) {              /* some lane needs an estimate */
        Mx X{0.0, -C[0], A[0], B[0], 0.0, D[0], -A[0]};
#pragma unroll
        for (int q = 1; q < L; ++q) X = mx_row(A[q], B[q], C[q], D[q], X);
        mx_norm(X);
        /* inclusive scan over the wave with DPP moves: shifts by 1, 2, 4, 8
         * within rows of 16 lanes, then the end of row r to row r + 1 (rows 1
         * and 3), then the end of row 1 to rows 2 and 3; the estimates need
         * not match any particular rounding */
        mx_scan_step<0x111>(X, (lane & 15) >= 1);
        mx_scan_step<0x112>(X, (lane & 15) >= 2);
        mx_scan_step<0x114>(X, (lane & 15) >= 4);
        mx_scan_step<0x118>(X, (lane & 15) >= 8);
        mx_scan_step<0x142>(X, (lane & 16) != 0);
        mx_scan_step<0x143>(X, lane >= 32);
        const double p = fma(X.a, ap, X.b), q = fma(X.c, ap, X.d), r = fma(X.e, ap, fma(X.g, bp, X.f));
        const double y = hd_div::rcp_refined(q);
        const int j = exact ? 0 : lane - m - 1;
        const double ea = __shfl(p * y, j, kSpecWave), eb = __shfl(r * y, j, kSpecWave);
        a0 = exact ? ap : ea;
        b0 = exact ? bp : eb;
    }
    /* warm-up rows, then the lane's own */
    double ca, cb, wa, wb, ra[L], rb[L];
    if (!plain) {
        hd_div::Range rg;
        ca = a0;
        cb = b0;
        double A4[4], B4[4], C4[4], D4[4];
        auto fetch = [&](int t0) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int t = t0 + u, p = (t & (L - 1)) * S + lane + (t >> LG);
                A4[u] = sA[p]; B4[u] = sB[p]; C4[u] = sC[p]; D4[u] = sD[p];
            }
        };
        fetch(0);
#pragma unroll
        for (int t0 = 0; t0 < kSpecWF; t0 += 4) { /* four rows, the next four on their way */
            double A3[4], B3[4], C3[4], D3[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) { A3[u] = A4[u]; B3[u] = B4[u]; C3[u] = C4[u]; D3[u] = D4[u]; }
            if (t0 + 4 < kSpecWF) fetch(t0 + 4);
#pragma unroll
            for (int u = 0; u < 4; ++u) thomas_row_warm(A3[u], B3[u], C3[u], D3[u], ca, cb);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (lane == 0) { ca = ap; cb = bp; }
        wa = ca;
        wb = cb;
#pragma unroll
        for (int q = 0; q < L; ++q) {
            thomas_row_rcp(A[q], B[q], C[q], D[q], ca, cb, rg);
            ra[q] = ca;
            rb[q] = cb;
        }
        plain = __any(act && !rows_ok(rg, ca, cb));
    }
    if (plain) {
        ca = a0;
        cb = b0;
#pragma unroll 1
        for (int t = 0; t < kSpecWF; ++t) {
            const int p = (t & (L - 1)) * S + lane + (t >> LG);
            if (lane * L - kSpecWF + t >= 0) thomas_row(sA[p], sB[p], sC[p], sD[p], ca, cb);
        }
        wa = ca;
        wb = cb;
#pragma unroll 1
        for (int t = 0; t < L; ++t) {
            const int p = t * S + own;
            thomas_row(sA[p], sB[p], sC[p], sD[p], ca, cb);
#pragma unroll
            for (int q = 0; q < L; ++q)
                if (q == t) { ra[q] = ca; rb[q] = cb; }
        }
    }
    /* exact verification against the predecessor's last row */
    {
        const double pa = lane_before(ca), pb = lane_before(cb);
        bool ok = lane == 0 || !act || (same_bits(wa, pa) && same_bits(wb, pb));
        unsigned long long bad = __ballot(!ok);
        if (bad) {
            if (fails && lane == 0) atomicAdd(fails, 1);
            /* where a failing lane's ap was right (ap depends on A, B, C only
             * and merges) its divisors are, and it redoes bp's chain alone */
            double e[L], y[L];
            hd_div::Range rd;
#pragma unroll
            for (int q = 0; q < L; ++q) {
                e[q] = A[q] * (q == 0 ? wa : ra[q - 1]) + B[q];
                y[q] = hd_div::rcp_refined(e[q]);
                rd.den(e[q]);
            }
            const bool mk = !nz && rd.den_ok();
            while (bad) {
                const int f = __ffsll((long long)bad) - 1; /* >= 1 */
                const double fa = readlane_f64(ca, f - 1), fb = readlane_f64(cb, f - 1);
                if (lane == f) {
                    if (same_bits(wa, fa)) {
                        hd_div::Range rn;
                        cb = fb;
#pragma unroll
                        for (int q = 0; q < L; ++q) {
                            cb = bp_known_e(A[q], D[q], cb, e[q], y[q], rn);
                            rb[q] = cb;
                        }
                        if (!(mk && rn.lo >= -720 && hd_div::finite(cb))) { /* outside the reciprocal form's range */
                            cb = fb;
#pragma unroll
                            for (int q = 0; q < L; ++q) {
                                cb = (D[q] - (A[q] * cb)) / e[q];
                                rb[q] = cb;
                            }
                        }
                    } else {
                        ca = fa;
                        cb = fb;
#pragma unroll
                        for (int q = 0; q < L; ++q) {
                            thomas_row(A[q], B[q], C[q], D[q], ca, cb);
                            ra[q] = ca;
                            rb[q] = cb;
                        }
                    }
                }
                const double na = readlane_f64(ca, f), nb = readlane_f64(cb, f);
                if (lane == f) ok = true;
                if (lane == f + 1) ok = !act || (same_bits(wa, na) && same_bits(wb, nb));
                bad = __ballot(!ok);
            }
        }
    }
    {
        const int ql = (n - 1) & (L - 1);
        double ea = ra[0], eb = rb[0];
#pragma unroll
        for (int q = 1; q < L; ++q)
            if (q == ql) { ea = ra[q]; eb = rb[q]; }
        ap = readlane_f64(ea, kl);
        bp = readlane_f64(eb, kl);
    }
    __syncthreads(); /* every lane has read C / D */
#pragma unroll
    for (int q = 0; q < L; ++q) {
        if (lane * L + q < n) {
            sC[q * S + own] = ra[q];
            sD[q * S + own] = rb[q];
        }
    }
    __syncthreads();
}

/* Forward elimination of the n rows of a sweep (at sm.pos(r) of the LDS
 * arrays), entering with the exact state (ap, bp) of the row before, which
 * is left as the state of row n - 1.  The factors ap / bp of the rows replace
 * C / D (after every lane has read them: speculating lanes keep their own
 * rows' factors in registers until the sweep is verified).  n <= 64 L; one
 * wave, uniform control; ends with a barrier.  fails: counts sweeps that
 * needed a repair. */
template <int MAXLG>
__device__ __forceinline__ void spec_forward(double* sA, double* sB, double* sC, double* sD, const SpecMap& sm, int n,
                                             double& ap, double& bp, int* fails = nullptr)
{
    if (n <= 0) return;
    if (sm.lg == 0) spec_forward_lg<0>(sA, sB, sC, sD, n, ap, bp, fails);
    else if (sm.lg == 1) spec_forward_lg<1>(sA, sB, sC, sD, n, ap, bp, fails);
    else if (MAXLG == 2 || sm.lg == 2) spec_forward_lg<2>(sA, sB, sC, sD, n, ap, bp, fails);
    else spec_forward_lg<3>(sA, sB, sC, sD, n, ap, bp, fails);
}

template <int LG>
__device__ __forceinline__ double spec_backward_lg(double* sAp, double* sBp, double* sX, int n, double x_in)
{
    constexpr int L = 1 << LG, S = spec_stride(LG), m = kSpecWB >> LG;
    constexpr SpecMap sm{LG};
    const int lane = threadIdx.x;
    const int kl = (n - 1) >> LG;
    /* identity factors (x = -0 + 1 x) where the warm-up reads past row n - 1 */
    if (n + lane < ((kl + 1) << LG) + kSpecWB) {
        const int p = sm.pos(n + lane);
        sAp[p] = 1.0;
        sBp[p] = -0.0;
    }
    __syncthreads();
    /* wave lane l takes the rows of forward lane kl - l, so that the chain
     * runs up the lanes */
    const bool act = lane <= kl;
    const int k = (act ? kl - lane : 0) + (kSpecWF >> LG);
    double oa[L], ob[L]; /* the lane's own factors */
#pragma unroll
    for (int q = 0; q < L; ++q) { oa[q] = sAp[q * S + k]; ob[q] = sBp[q * S + k]; }
    const bool exact = lane <= m;
    double cx = x_in;
    if (n > kSpecWB + L) {
        double al = oa[L - 1], be = ob[L - 1];
#pragma unroll
        for (int q = L - 2; q >= 0; --q) {
            be = fma(oa[q], be, ob[q]);
            al = oa[q] * al;
        }
        /* inclusive scan of the affine maps, DPP moves as in the forward sweep */
        aff_scan_step<0x111>(al, be, (lane & 15) >= 1);
        aff_scan_step<0x112>(al, be, (lane & 15) >= 2);
        aff_scan_step<0x114>(al, be, (lane & 15) >= 4);
        aff_scan_step<0x118>(al, be, (lane & 15) >= 8);
        aff_scan_step<0x142>(al, be, (lane & 16) != 0);
        aff_scan_step<0x143>(al, be, lane >= 32);
        const double est = __shfl(fma(al, x_in, be), exact ? 0 : lane - m - 1, kSpecWave);
        cx = exact ? x_in : est;
    }
    /* warm-up: the 32 rows above the lane's, last first */
    {
        double a8[8], b8[8];
        auto fetch = [&](int t0) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int t = kSpecWB - 1 - t0 - u, p = (t & (L - 1)) * S + k + 1 + (t >> LG);
                a8[u] = sAp[p];
                b8[u] = sBp[p];
            }
        };
        fetch(0);
#pragma unroll
        for (int t0 = 0; t0 < kSpecWB; t0 += 8) { /* eight rows, the next eight on their way */
            double a[8], b[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) { a[u] = a8[u]; b[u] = b8[u]; }
            if (t0 + 8 < kSpecWB) fetch(t0 + 8);
#pragma unroll
            for (int u = 0; u < 8; ++u) cx = b[u] + (a[u] * cx);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    const double w = cx;
    auto rows = [&]() {
#pragma unroll
        for (int q = L - 1; q >= 0; --q) {
            cx = ob[q] + (oa[q] * cx);
            sX[q * S + k] = cx;
        }
    };
    if (act) rows();
    {
        const double px = lane_before(cx);
        bool ok = exact || !act || same_bits(w, px);
        unsigned long long bad = __ballot(!ok);
        while (bad) {
            const int f = __ffsll((long long)bad) - 1;
            const double fx = readlane_f64(cx, f - 1);
            if (lane == f) {
                cx = fx;
                rows();
            }
            const double nx = readlane_f64(cx, f);
            if (lane == f) ok = true;
            if (lane == f + 1) ok = exact || !act || same_bits(w, nx);
            bad = __ballot(!ok);
        }
    }
    const double x0 = readlane_f64(cx, kl);
    __syncthreads();
    return x0;
}

/* Back substitution over the n rows of a sweep, last first, given x of the
 * row after them; x_r goes to sX[sm.pos(r)].  Returns x of row 0 (x_in when
 * n <= 0). */
template <int MAXLG>
__device__ __forceinline__ double spec_backward(double* sAp, double* sBp, double* sX, const SpecMap& sm, int n,
                                                double x_in)
{
    if (n <= 0) return x_in;
    if (sm.lg == 0) return spec_backward_lg<0>(sAp, sBp, sX, n, x_in);
    if (sm.lg == 1) return spec_backward_lg<1>(sAp, sBp, sX, n, x_in);
    if (MAXLG == 2 || sm.lg == 2) return spec_backward_lg<2>(sAp, sBp, sX, n, x_in);
    return spec_backward_lg<3>(sAp, sBp, sX, n, x_in);
}

} // namespace hd_spec

#endif
