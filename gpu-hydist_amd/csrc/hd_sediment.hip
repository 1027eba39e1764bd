/*
 * hd_sediment.hip -- suspended-sediment sweep and bed change
 * (Sediment_Transport.cu), gfx950.
 *
 * Per half-step with t >= sediment_start: VTH + hesoK (one thread per cell),
 * the concentration rows of the sweep direction (one thread per interior cell
 * of each wet run), one lane per line for the Thomas solve with the
 * extraction into tFS, then FS = tFS.  Bed change: Calculate_Qb then
 * _bed_load, one thread per cell.  Formulas follow the cited reference lines
 * in the same operation order (contraction off).
 */
#include "hd_edges.h"
#include "hd_internal.h"
#include "hd_thomas.h"

namespace {

/* Cell (i, j) of a thread of a block of 256 over the context's active 64-column row tiles
 * (tiles holding or bordering a cell with khouot != 2): outside them the
 * sediment kernels that run by tiles have reached a fixed point once they
 * have run over the whole grid, which the caller arranges. */
__device__ __forceinline__ bool tile_cell(const HdDevG& d, int& i, int& j, int first = 0)
{
    const int t = xcd_block((int)blockIdx.x - first, (int)gridDim.x - first) * 4 + wave_in_block();
    if (!active_tile(d, t, i, j)) return false;
    j += threadIdx.x & 63;
    return j < d.M + 3 && i < d.N + 3;
}

/* source_chs, Sediment_Transport.cu:12-49. */
__device__ double source_chs(const hd_params& P, double wsm, double Zf, double fs, double fw, double vth, double h_moi)
{
    double toee = P.Toe, todd = P.Tod, S = 0;
    double tob = P.ro * fw * (vth * vth);
    if (h_moi > P.ghtoe) toee = P.Toe * (1 + P.hstoe * ((h_moi - P.ghtoe)));
    if (tob > toee) S = P.Mbochat / P.ros * (tob - toee) / toee;
    else if (tob < todd) {
        double Pd = 1 - (tob / todd);
        double beta = 1 + (Zf / (1.25 + 4.75 * hd_pow(Pd, 2.5)));
        double Cb = beta * fs;
        S = -wsm * Cb * Pd;
    }
    return S;
}

/* The fast forms of the rows below take each quotient from the refined
 * reciprocal of its divisor (hd_fastdiv.h) and the powers and logarithms
 * without their special arguments; FsGuard collects what that takes for
 * granted, and a wave in which a lane fails it evaluates the plain forms. */
struct FsGuard {
    hd_div::Range g;
    bool bad = false;
    __device__ __forceinline__ bool ok() const { return !bad && g.lo >= -800 && g.den_ok(); }
};

/* wave-uniform values of the rows: reciprocals of the case constants */
struct FsConst {
    double sqrtg, Ufr2, hT, cd;              /* sqrt(g), Ufr^2, dT/2, 0.015 dm */
    double yKs, yUfr2, yhT, ydX2, ydY2;      /* refined reciprocals */
    bool ok;                                 /* constants positive, within 2^-50 .. 2^50 */
};

__device__ __forceinline__ FsConst fs_const(const HdDevG& d)
{
    const hd_params& P = d.P;
    FsConst k;
    k.sqrtg = sqrt(P.g);
    k.Ufr2 = P.Ufr * P.Ufr;
    k.hT = P.dT * 0.5;
    k.cd = 0.015 * P.dm;
    k.yKs = hd_div::rcp_refined(P.Ks);
    k.yUfr2 = hd_div::rcp_refined(k.Ufr2);
    k.yhT = hd_div::rcp_refined(k.hT);
    k.ydX2 = hd_div::rcp_refined(P.dX2);
    k.ydY2 = hd_div::rcp_refined(P.dY2);
    const double c[] = {P.Ks, k.Ufr2, k.hT, P.dX2, P.dY2, P.dXbp, P.dYbp, P.wss, P.g, k.cd, d.Dxr_m03};
    k.ok = true;
#pragma unroll
    for (double v : c) k.ok = k.ok && v > 0x1p-50 && v < 0x1p50;
    return k;
}

template <bool FAST>
__device__ __forceinline__ double fs_div(double n, double e, double y)
{
    return FAST ? hd_div::quot_pos(n, e, y) : n / e;
}
template <bool FAST>
__device__ __forceinline__ double fs_rcp(double e)
{
    return FAST ? hd_div::rcp_refined(e) : 0.0;
}

/* The source term S of a cell with depth hm, concentration fs and speed vth
 * (source_chs, or source_nchs, Sediment_Transport.cu:52-60) and its Zf (0
 * unless fs > thr), as the rows (Sediment_Transport.cu:90-100) and the bed
 * change (:490-500) evaluate them.  The fast form's quotients are in range
 * for constants within 2^-50 .. 2^50, divisors within 2^-100 .. 2^100 and
 * the numerators that the guard takes; the clamp of Tx at 0 would hide a
 * NaN, so its numerator is tested by itself. */
template <bool FAST>
__device__ __forceinline__ double fs_source(const HdDevG& d, const FsConst& K, int ketdinh, double thr, double hm,
                                            double fs, double vth, double fw, double& Zf, FsGuard& G)
{
    const hd_params& P = d.P;
    const double xl = fs_div<FAST>(12 * hm, P.Ks, K.yKs);
    const double c = 18 * (FAST ? hd_log_core(xl) : hd_log(xl));
    const double nu = K.sqrtg * fabs(vth);
    const double Uf = FAST ? hd_div::quot(nu, c, hd_div::rcp_refined(c)) : nu / c;
    const double z = 1 - fs;
    const double wsm = P.wss * (FAST ? hd_pow_core(fabs(z), 4) : hd_pow(z, 4));
    Zf = 0;
    const double ez = 0.4 * (Uf + 2 * wsm);
    if (fs > thr) Zf = fs_div<FAST>(wsm, ez, fs_rcp<FAST>(ez));
    if (FAST) {
        G.bad = G.bad || !(hm > 0) || z == 0;
        G.g.den(hm); G.g.den(c); G.g.den(z); G.g.den(ez);
        G.g.num(vth);
    }
    if (ketdinh) return source_chs(P, wsm, Zf, fs, fw, vth, hm);
    const double gamac = 0.434 + 5.975 * Zf + 2.888 * Zf * Zf;
    const double nt = Uf * Uf - K.Ufr2;
    const double Tx = fmax(0.0, fs_div<FAST>(nt, K.Ufr2, K.yUfr2));
    double pt = 0.0;
    if (FAST) {
        G.bad = G.bad || !(nt < 0x1p200);
        G.g.den(Tx);
        if (__any(Tx > 0)) pt = Tx > 0 ? hd_pow_core(Tx, 1.5) : 0.0;
    } else {
        pt = hd_pow(Tx, 1.5);
    }
    const double e5 = 0.05 * hm;
    const double Cac = fs_div<FAST>(K.cd * pt * d.Dxr_m03, e5, fs_rcp<FAST>(e5));
    return wsm * (Cac - gamac * fs);
}

/* Find_VTH (Sediment_Transport.cu:541-568) and hesoK (:508-539).  Bound by
 * the chain of its loads (view, tile, fields): all fields are loaded at
 * once, 5.7 us on a 980 x 1048 river grid against 7.1 with the loads behind
 * the tests.
 * bnd (with tiles): the launch has one workgroup more, the first, which
 * writes the half-step's boundary values, a wave an edge, as k_boundary does;
 * nothing here reads those.  A step on a frozen flow, bed change included, same
 * grid: 69.8 us with two k_boundary launches, 64.1 without. */
__global__ void __launch_bounds__(256) k_vth_hesok(const HdDev* __restrict__ dv, int tiled, int bnd)
{
    const HdDevG& d = dev_view(dv);
    int j, i;
    if (bnd && blockIdx.x == 0) {
        boundary_series<64, 4>(d, wave_in_block(), threadIdx.x & 63);
        return;
    }
    if (tiled) {
        if (!tile_cell(d, i, j, bnd)) return;
    } else {
        j = blockIdx.x * blockDim.x + threadIdx.x;
        i = blockIdx.y;
    }
    int N = d.N, M = d.M, W = d.W;
    const hd_params& P = d.P;
    if (i < 1 || j < 1 || j > M || i > N) return;
    const int pos = i * W + j;
    /* one round of loads */
    const double u0 = d.t_u[pos], um = d.t_u[pos - W], v0 = d.t_v[pos], vm = d.t_v[pos - 1];
    const double hu = d.Htdu[pos], hv = d.Htdv[pos], hm = d.H_moi[pos], hz = d.htaiz[pos];
    const double h0 = d.h[pos], hx = d.h[pos - 1], hy = d.h[pos - W];
    if (i >= 2 && j >= 2) {
        double vth = 0;
        if ((hz > P.NANGDAY) && (hm > P.H_TINH)) {
            double ut = (u0 + um) * 0.5;
            double vt = (v0 + vm) * 0.5;
            vth = sqrt(ut * ut + vt * vt);
        }
        d.VTH[pos] = vth;
    }
    const double sg = 5.93 * sqrt(P.g);
    if (hu > 0) {
        double Cz = 18 * hd_log(12 * hu / P.Ks);
        double kx = sg * (hx + h0) * 0.25 * fabs(u0) / Cz;
        d.Kx[pos] = fmin(100.0, fmax(5.0, kx));
    }
    if (hv > 0) {
        double Cz = 18 * hd_log(12 * hv / P.Ks);
        double ky = sg * (hy + h0) * 0.25 * fabs(v0) / Cz;
        d.Ky[pos] = fmin(100.0, fmax(5.0, ky));
    }
}

__device__ __forceinline__ void wall_flags2(const HdDevG& d, bool isJ, int line, int first, int last, bool& br1, bool& br2)
{
    int W = d.W;
    const double* h = d.h;
    double ND = d.P.NANGDAY;
    if (isJ) { /* locate_segment_u, column line */
        br1 = (first > 2) || ((first == 2) && ((h[1 * W + line] + h[1 * W + line - 1]) * 0.5 == ND));
        br2 = (last < d.N) || ((last == d.N) && ((h[d.N * W + line] + h[d.N * W + line - 1]) * 0.5 == ND));
    } else {   /* locate_segment_v, row line */
        br1 = (first > 2) || ((first == 2) && ((h[line * W + first - 1] + h[(line - 1) * W + first - 1]) * 0.5 == ND));
        br2 = (last < d.M) || ((last == d.M) && ((h[line * W + last] + h[(line - 1) * W + last]) * 0.5 == ND));
    }
}

struct FsRow {
    double A, B, C, D;
};

/* What a row reads: along the line the velocity, the face depth and K at the
 * cell and the one before (u, hu, k; suffix m), across it the same (v, hv,
 * kv) and the depth and concentration at the neighbours. */
struct FsRaw {
    double u0, um, hu0, hum, k0, km;
    double v0, vm, hv0, hvm, kv0, kvm;
    double h0, hp1, hp2, hm1, hm2;
    double f0, fp, fm;
    double vth, fw;
};

/* The run's ends: the first / last row takes its end cell's coefficient into
 * B (wall, or no flow there), else its concentration into D. */
struct FsEnds {
    bool w1, w2, c2; /* c2: the end copy's test at the last cell */
    double f1, f2;
};

template <bool isJ>
__device__ __forceinline__ FsEnds fs_ends(const HdDevG& d, int line, int first, int last, bool br1, bool br2)
{
    const int W = d.W;
    const double* tq = isJ ? d.t_u : d.t_v;
    const int p1 = isJ ? first * W + line : line * W + first, p2 = isJ ? last * W + line : line * W + last;
    FsEnds e;
    const double q1 = tq[p1], q2 = tq[p2];
    e.f1 = d.FS[p1];
    e.f2 = d.FS[p2];
    e.w1 = br1 || q1 == 0;
    e.c2 = br2 || q2 == 0;
    e.w2 = isJ ? (br2 && q2 == 0) : e.c2; /* as written */
    return e;
}

template <bool isJ>
__device__ __forceinline__ FsRaw fs_load(const HdDevG& d, int i, int j)
{
    const int W = d.W, pos = i * W + j, s = isJ ? W : 1, t = isJ ? 1 : W;
    const double *u = isJ ? d.t_u : d.t_v, *v = isJ ? d.t_v : d.t_u;
    const double *hu = isJ ? d.Htdu : d.Htdv, *hv = isJ ? d.Htdv : d.Htdu;
    const double *ku = isJ ? d.Kx : d.Ky, *kv = isJ ? d.Ky : d.Kx;
    const double *H = d.H_moi, *F = d.FS;
    FsRaw r;
    r.u0 = u[pos]; r.um = u[pos - s]; r.hu0 = hu[pos]; r.hum = hu[pos - s]; r.k0 = ku[pos]; r.km = ku[pos - s];
    r.v0 = v[pos]; r.vm = v[pos - t]; r.hv0 = hv[pos]; r.hvm = hv[pos - t]; r.kv0 = kv[pos]; r.kvm = kv[pos - t];
    r.h0 = H[pos]; r.hp1 = H[pos + t]; r.hp2 = H[pos + 2 * t]; r.hm1 = H[pos - t]; r.hm2 = H[pos - 2 * t];
    r.f0 = F[pos]; r.fp = F[pos + t]; r.fm = F[pos - t];
    r.vth = d.VTH[pos];
    r.fw = d.Fw[pos];
    return r;
}

/* two neighbouring elements in one load, aligned to 8 bytes */
typedef double hd_pair __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ hd_pair ld2_off(HD_GLOBAL_AS const double* p, long base, unsigned off)
{
    return *(HD_GLOBAL_AS const hd_pair*)((HD_GLOBAL_AS const char*)(p + base) + off);
}

/* fs_load of 64 successive cells, lane l's at element base + off / 8 (off
 * the lane's offset along the line); before: the base of the cell before
 * lane 0's.  A column's cells lie in 64 cache lines, and a load of 64 lines
 * keeps the address unit for 64 cycles: its values along the line come from
 * the lane before, and neighbours across it in pairs, 12 loads in place of
 * 22. */
template <bool isJ>
__device__ __forceinline__ FsRaw fs_load_off(const HdDevG& d, int ketdinh, long b, long before, unsigned o)
{
    const long W = d.W;
    FsRaw r;
    r.fw = 0;
    if (isJ) {
        r.u0 = ld_off(d.t_u, b, o); r.hu0 = ld_off(d.Htdu, b, o); r.k0 = ld_off(d.Kx, b, o);
        const double xu = ld_off(d.t_u, before, 0), xh = ld_off(d.Htdu, before, 0), xk = ld_off(d.Kx, before, 0);
        const hd_pair v = ld2_off(d.t_v, b - 1, o), hv = ld2_off(d.Htdv, b - 1, o), kv = ld2_off(d.Ky, b - 1, o);
        const hd_pair ha = ld2_off(d.H_moi, b - 2, o), hb = ld2_off(d.H_moi, b, o);
        const hd_pair f = ld2_off(d.FS, b - 1, o);
        r.hp2 = ld_off(d.H_moi, b + 2, o);
        r.fp = ld_off(d.FS, b + 1, o);
        r.vth = ld_off(d.VTH, b, o);
        if (ketdinh) r.fw = ld_off(d.Fw, b, o);
        r.vm = v.x; r.v0 = v.y; r.hvm = hv.x; r.hv0 = hv.y; r.kvm = kv.x; r.kv0 = kv.y;
        r.hm2 = ha.x; r.hm1 = ha.y; r.h0 = hb.x; r.hp1 = hb.y;
        r.fm = f.x; r.f0 = f.y;
        r.um = xu; r.hum = xh; r.km = xk; /* lane 0's; fs_before gives the others theirs */
    } else {
        const hd_pair u = ld2_off(d.t_v, b - 1, o), hu = ld2_off(d.Htdv, b - 1, o), ku = ld2_off(d.Ky, b - 1, o);
        r.v0 = ld_off(d.t_u, b, o); r.vm = ld_off(d.t_u, b - W, o);
        r.hv0 = ld_off(d.Htdu, b, o); r.hvm = ld_off(d.Htdu, b - W, o);
        r.kv0 = ld_off(d.Kx, b, o); r.kvm = ld_off(d.Kx, b - W, o);
        r.h0 = ld_off(d.H_moi, b, o);
        r.hp1 = ld_off(d.H_moi, b + W, o); r.hp2 = ld_off(d.H_moi, b + 2 * W, o);
        r.hm1 = ld_off(d.H_moi, b - W, o); r.hm2 = ld_off(d.H_moi, b - 2 * W, o);
        r.f0 = ld_off(d.FS, b, o); r.fp = ld_off(d.FS, b + W, o); r.fm = ld_off(d.FS, b - W, o);
        r.vth = ld_off(d.VTH, b, o);
        if (ketdinh) r.fw = ld_off(d.Fw, b, o);
        r.um = u.x; r.u0 = u.y; r.hum = hu.x; r.hu0 = hu.y; r.km = ku.x; r.k0 = ku.y;
    }
    return r;
}

template <bool isJ>
__device__ __forceinline__ void fs_before(FsRaw& r)
{
    if (!isJ) return;
    r.um = hd_spec::dpp_f64<0x138, 0xF>(r.um, r.u0);
    r.hum = hd_spec::dpp_f64<0x138, 0xF>(r.hum, r.hu0);
    r.km = hd_spec::dpp_f64<0x138, 0xF>(r.km, r.k0);
}

/* One concentration row from its loads: _FSj_calculate__mactrix_coeff
 * (Sediment_Transport.cu:205-302, column lines, gamav before Zf, as written)
 * or _FSi_calculate__mactrix_coeff (:62-165, row lines); is1 / is2: the
 * run's first / last row.  Quotients that differ in sign only are taken
 * once; every other operation is the reference's, in its order. */
template <bool isJ, bool FAST>
__device__ __forceinline__ FsRow fs_eval(const HdDevG& d, const FsConst& K, const FsRaw& r, const FsEnds& E, bool src,
                                         int ketdinh, bool is1, bool is2, FsGuard& G)
{
    const hd_params& P = d.P;
    const double dL2 = isJ ? P.dX2 : P.dY2, dLb = isJ ? P.dXbp : P.dYbp;
    const double dC2 = isJ ? P.dY2 : P.dX2, dCb = isJ ? P.dYbp : P.dXbp;
    const double yL2 = isJ ? K.ydX2 : K.ydY2, yC2 = isJ ? K.ydY2 : K.ydX2;
    double Zf;
    double S = fs_source<FAST>(d, K, ketdinh, 0.00001, r.h0, r.f0, r.vth, r.fw, Zf, G);
    if (!src) S = 0;
    const double Zg = isJ ? 0.0 : Zf;
    const double gamav = 0.98 - 0.198 * Zg + 0.032 * Zg * Zg;
    const double na = gamav * 0.5 * (r.u0 + r.um);
    const double qa = fs_div<FAST>(na, dL2, yL2);
    const double e1 = r.h0 * dLb, y1 = fs_rcp<FAST>(e1);
    const double n0 = r.hu0 * r.k0, nm = r.hum * r.km;
    const double A = -qa - fs_div<FAST>(nm, e1, y1);
    const double C = qa - fs_div<FAST>(n0, e1, y1);
    double B = P.HaiChiadT + fs_div<FAST>(n0 + nm, e1, y1);
    double p = 0, q = 0;
    if (r.hm1 > P.H_TINH && r.hp2 > P.H_TINH) p = r.fp - r.f0;
    if (r.hm2 > P.H_TINH && r.hp1 > P.H_TINH) q = r.f0 - r.fm;
    const double e2 = r.h0 * dCb;
    p = fs_div<FAST>(1.0, e2, fs_rcp<FAST>(e2)) * (r.hv0 * r.kv0 * p - r.hvm * r.kvm * q);
    q = 0;
    const double nq = r.fp - r.fm;
    if (r.hm2 > P.H_TINH && r.hp2 > P.H_TINH) q = (r.v0 + r.vm) * 0.5 * fs_div<FAST>(nq, dC2, yC2) * gamav;
    double D = fs_div<FAST>(r.f0, K.hT, K.yhT) - q + p + fs_div<FAST>(S, r.h0, fs_rcp<FAST>(r.h0));
    if (is1) {
        if (E.w1) B += A;
        else D -= A * E.f1;
    }
    if (is2) {
        if (E.w2) B += C;
        else D -= C * E.f2;
    }
    if (FAST) {
        G.g.num(na); G.g.num(n0); G.g.num(nm); G.g.num(nq); G.g.num(r.f0); G.g.num(S);
        G.bad = G.bad || !hd_div::finite(A) || !hd_div::finite(B) || !hd_div::finite(C) || !hd_div::finite(D);
    }
    FsRow w;
    w.A = A; w.B = B; w.C = C; w.D = D;
    return w;
}

/* The row of cell (i, j) of run [first, last], plain. */
template <bool isJ>
__device__ FsRow fs_row(const HdDevG& d, double t, double s_start, int ketdinh, int i, int j, int first, int last,
                        bool br1, bool br2)
{
    const int k = isJ ? i : j, line = isJ ? j : i;
    FsConst K;
    K.sqrtg = sqrt(d.P.g);
    K.Ufr2 = d.P.Ufr * d.P.Ufr;
    K.hT = d.P.dT * 0.5;
    K.cd = 0.015 * d.P.dm;
    FsGuard G;
    return fs_eval<isJ, false>(d, K, fs_load<isJ>(d, i, j), fs_ends<isJ>(d, line, first, last, br1, br2),
                               !(t < s_start), ketdinh, k == first + 1, k == last - 1, G);
}

/* Concentration rows: _FSj_calculate__mactrix_coeff (Sediment_Transport.cu:205-302,
 * column lines, gamav before Zf and && at the last row, as written) or
 * _FSi_calculate__mactrix_coeff (:62-165, row lines).  Row of cell k sits at
 * line*tw + k. */
template <bool isJ>
__global__ void __launch_bounds__(256) k_fs_coef(const HdDev* __restrict__ dv, double s_start, int ketdinh)
{
    const HdDevG& d = dev_view(dv);
    const double* tdev = d.tdev;
    __shared__ int s_moc[64];
    __shared__ int s_dau[64][24];
    __shared__ int s_cuoi[64][24];
    int N = d.N, M = d.M, SL = d.SL;
    int tx = threadIdx.x, ty = threadIdx.y;
    int j0 = blockIdx.x * 64, i0 = blockIdx.y * 16;
    int tid = ty * 64 + tx;
    int sidx = 3, eidx = isJ ? M - 1 : N - 1;
    if (isJ) {
        for (int t = tid; t < 64; t += 256) {
            int L = j0 + t;
            s_moc[t] = (L >= sidx && L <= eidx) ? min(d.mocj[L], SL) : 0;
        }
        __syncthreads();
        for (int t = tid; t < 64 * SL; t += 256) {
            int c = t / SL, s = t % SL;
            if (s < s_moc[c]) { s_dau[c][s] = d.dauj[(j0 + c) * SL + s]; s_cuoi[c][s] = d.cuoij[(j0 + c) * SL + s]; }
        }
    } else {
        for (int t = tid; t < 16; t += 256) {
            int L = i0 + t;
            s_moc[t] = (L >= sidx && L <= eidx) ? min(d.moci[L], SL) : 0;
        }
        __syncthreads();
        for (int t = tid; t < 16 * SL; t += 256) {
            int c = t / SL, s = t % SL;
            if (s < s_moc[c]) { s_dau[c][s] = d.daui[(i0 + c) * SL + s]; s_cuoi[c][s] = d.cuoii[(i0 + c) * SL + s]; }
        }
    }
    __syncthreads();
    int j = j0 + tx;
    if (j > M) return;
    const double t = tdev[0];
    const int tw = 2 * (N > M ? N : M) + 4;
    for (int r = ty; r < 16; r += 4) {
        int i = i0 + r;
        if (i > N) break;
        int li = isJ ? tx : r;
        int k = isJ ? i : j;
        int line = isJ ? j : i;
        int first = 0, last = 0, n = s_moc[li];
        bool found = false;
        for (int s = 0; s < n; ++s) {
            if (s_dau[li][s] <= k && k <= s_cuoi[li][s]) { first = s_dau[li][s]; last = s_cuoi[li][s]; found = true; break; }
        }
        if (!found || last < first + 2 || k < first + 1 || k > last - 1) continue;
        bool br1, br2;
        wall_flags2(d, isJ, line, first, last, br1, br2);
        FsRow w = fs_row<isJ>(d, t, s_start, ketdinh, i, j, first, last, br1, br2);
        double A = w.A, B = w.B, C = w.C, D = w.D;
        size_t o = (size_t)line * tw + k;
        d.AA[o] = A; d.BB[o] = B; d.CC[o] = C; d.DD[o] = D;
    }
}

/* tridiagSolver (jump 1) + FSj/FSi_extract_solution (Sediment_Transport.cu:
 * 305-338 / 168-202), one lane per line.  Runs with last - first < 2 have no
 * rows and are skipped. */
template <bool isJ>
__global__ void __launch_bounds__(64) k_fs_solve(const HdDev* __restrict__ dv)
{
    const HdDevG& d = dev_view(dv);
    int N = d.N, M = d.M, W = d.W, SL = d.SL;
    int line = 3 + blockIdx.x * blockDim.x + threadIdx.x;
    if (line > (isJ ? M - 1 : N - 1)) return;
    const int tw = 2 * (N > M ? N : M) + 4;
    int nseg = isJ ? d.mocj[line] : d.moci[line];
    if (nseg > SL) nseg = SL;
    const int* dau = (isJ ? d.dauj : d.daui) + line * SL;
    const int* cuoi = (isJ ? d.cuoij : d.cuoii) + line * SL;
    size_t base = (size_t)line * tw;
    const double *AA = d.AA + base, *BB = d.BB + base, *CC = d.CC + base, *DD = d.DD + base;
    double *Ap = d.Ap + base, *Bp = d.Bp + base;
    auto at = [&](int k) -> size_t { return isJ ? (size_t)k * W + line : (size_t)line * W + k; };
    for (int s = 0; s < nseg; ++s) {
        int first = dau[s], last = cuoi[s];
        if (last < first + 2) continue;
        bool br1, br2;
        wall_flags2(d, isJ, line, first, last, br1, br2);
        int sn = last - first - 2;
        int o = first + 1;
        double x;
        if (sn == 0) x = DD[o] / BB[o];
        else {
            double ap = -CC[o] / BB[o], bp = DD[o] / BB[o];
            Ap[o] = ap; Bp[o] = bp;
            for (int r = 1; r < sn; ++r) {
                double a = AA[o + r];
                double e = a * ap + BB[o + r];
                double nap = -CC[o + r] / e;
                double nbp = (DD[o + r] - (a * bp)) / e;
                ap = nap; bp = nbp;
                Ap[o + r] = ap; Bp[o + r] = bp;
            }
            double a = AA[o + sn];
            x = (DD[o + sn] - (a * bp)) / (BB[o + sn] + (a * ap));
        }
        double vfirst = 0, vlast = 0;
        for (int r = sn; r >= 0; --r) {
            if (r < sn) x = Bp[o + r] + (Ap[o + r] * x);
            double v = x;
            if (v < 0) v = d.P.NDnen;
            d.tFS[at(o + r)] = v;
            if (r == 0) vfirst = v;
            if (r == sn) vlast = v;
        }
        /* end copies (FSj: t_u at first / last; FSi: t_v at first / last) */
        const double* tq = isJ ? d.t_u : d.t_v;
        if ((br1) || (tq[at(first)] == 0)) d.tFS[at(first)] = vfirst;
        else d.tFS[at(first)] = d.FS[at(first)];
        if ((br2) || (tq[at(last)] == 0)) d.tFS[at(last)] = vlast;
        else d.tFS[at(last)] = d.FS[at(last)];
    }
}

/* Fused concentration sweep, one wave per line: rows of 64 interior cells
 * at a time in parallel into LDS, lane 0 runs the Thomas recurrence
 * (UVZSolver_multithread.cu:203-228, jump 1) over them, then back
 * substitution and the extraction into tFS with the end copies
 * (Sediment_Transport.cu:305-338 / 168-202), lanes in parallel. */
template <bool isJ>
__global__ void __launch_bounds__(64) k_fs_line(const HdDev* __restrict__ dv, double s_start, int ketdinh)
{
    const HdDevG& d = dev_view(dv);
    const double* tdev = d.tdev;
    constexpr int CH = 64;
    constexpr int kCap = 2048;
    __shared__ double sA[CH], sB[CH], sC[CH], sD[CH];
    __shared__ double sAp[kCap], sBp[kCap];
    int N = d.N, M = d.M, W = d.W, SL = d.SL;
    int line = 3 + blockIdx.x;
    if (line > (isJ ? M - 1 : N - 1)) return;
    int lane = threadIdx.x;
    const int tw = 2 * (N > M ? N : M) + 4;
    const double t = tdev[0];
    int nseg = isJ ? d.mocj[line] : d.moci[line];
    if (nseg > SL) nseg = SL;
    const int* dau = (isJ ? d.dauj : d.daui) + line * SL;
    const int* cuoi = (isJ ? d.cuoij : d.cuoii) + line * SL;
    double* gAp = d.Ap + (size_t)line * tw;
    double* gBp = d.Bp + (size_t)line * tw;
    auto at = [&](int k) -> size_t { return isJ ? (size_t)k * W + line : (size_t)line * W + k; };
    for (int s = 0; s < nseg; ++s) {
        int first = dau[s], last = cuoi[s];
        if (last < first + 2) continue;
        bool br1, br2;
        wall_flags2(d, isJ, line, first, last, br1, br2);
        int sn = last - first - 2;
        int k0 = first + 1;
        double* oAp = gAp + k0;
        double* oBp = gBp + k0;
        double ap = 0, bp = 0, xs = 0;
        for (int c0 = 0; c0 <= sn; c0 += CH) {
            int r = c0 + lane;
            if (r <= sn) {
                int k = k0 + r;
                int i = isJ ? k : line, j = isJ ? line : k;
                FsRow w = fs_row<isJ>(d, t, s_start, ketdinh, i, j, first, last, br1, br2);
                sA[lane] = w.A; sB[lane] = w.B; sC[lane] = w.C; sD[lane] = w.D;
            }
            __syncthreads();
            if (lane == 0) {
                int re = c0 + CH - 1;
                if (re > sn) re = sn;
                for (int q = c0; q <= re; ++q) {
                    double A = sA[q - c0], B = sB[q - c0], C = sC[q - c0], D = sD[q - c0];
                    if (q == 0 && sn == 0) xs = D / B;
                    else if (q == 0) { ap = -C / B; bp = D / B; }
                    else if (q < sn) {
                        double e = A * ap + B;
                        double nap = -C / e;
                        double nbp = (D - (A * bp)) / e;
                        ap = nap; bp = nbp;
                    } else xs = (D - (A * bp)) / (B + (A * ap));
                    if (q < sn) {
                        if (q < kCap) { sAp[q] = ap; sBp[q] = bp; }
                        else { oAp[q] = ap; oBp[q] = bp; }
                    }
                }
            }
            __syncthreads();
        }
        if (lane == 0) {
            double x = xs;
            if (sn < kCap) sBp[sn] = x; else oBp[sn] = x;
            for (int q = sn - 1; q >= 0; --q) {
                double apq = q < kCap ? sAp[q] : oAp[q];
                double bpq = q < kCap ? sBp[q] : oBp[q];
                x = bpq + (apq * x);
                if (q < kCap) sBp[q] = x; else oBp[q] = x;
            }
        }
        __syncthreads();
        for (int q = lane; q <= sn; q += 64) {
            double v = q < kCap ? sBp[q] : oBp[q];
            if (v < 0) v = d.P.NDnen;
            d.tFS[at(k0 + q)] = v;
        }
        __syncthreads();
        if (lane == 0) {
            double vfirst = d.tFS[at(k0)], vlast = d.tFS[at(last - 1)];
            const double* tqq = isJ ? d.t_u : d.t_v;
            if ((br1) || (tqq[at(first)] == 0)) d.tFS[at(first)] = vfirst;
            else d.tFS[at(first)] = d.FS[at(first)];
            if ((br2) || (tqq[at(last)] == 0)) d.tFS[at(last)] = vlast;
            else d.tFS[at(last)] = d.FS[at(last)];
        }
        __syncthreads();
    }
}

/* The FS sweep with one wave per wet run from the packed run tables (runs_u
 * for the column sweep FSj, runs_v for the row sweep FSi), lines 3 .. M-1 /
 * N-1 as the reference launches them.  Rows are assembled by the 64 lanes in
 * chunks of 256 (four per lane) into LDS; lane 0 carries the Thomas
 * recurrence (the same operations in the same order as k_fs_line and the
 * reference's tridiagSolver); factors of all but the last chunk go to the
 * run's slice of Ap/Bp.  The end copies use the clamped first / last
 * solutions kept in LDS. */
template <bool isJ>
__global__ void __launch_bounds__(64) k_fs_run(const HdDev* __restrict__ dv, double s_start, int ketdinh)
{
    const HdDevG& d = dev_view(dv);
    constexpr int RW = 256;
    __shared__ double sA[RW], sB[RW], sC[RW], sD[RW];
    __shared__ double sV[2]; /* clamped x of the first and last row */
    const int N = d.N, M = d.M, W = d.W;
    const int lane = threadIdx.x;
    const int tw = 2 * (N > M ? N : M) + 4;
    const int lmax = isJ ? M - 1 : N - 1;
    const int cap = (isJ ? M + 3 : N + 3) * d.SL;
    const int cnt = d.run_cnt[isJ ? 0 : 1] < cap ? d.run_cnt[isJ ? 0 : 1] : cap;
    const int4* runs = isJ ? d.runs_u : d.runs_v;
    const double t = d.tdev[0];
    const RunSlice sl = run_slice(cnt);
    for (int ri = sl.start; ri < sl.end; ri += sl.step) {
        const int4 rn = runs[ri];
        const int line = rn.x, first = rn.y, last = rn.z;
        if (line < 3 || line > lmax || last < first + 2) continue;
        auto at = [&](int k) -> size_t { return isJ ? (size_t)k * W + line : (size_t)line * W + k; };
        bool br1, br2;
        wall_flags2(d, isJ, line, first, last, br1, br2);
        const int sn = last - first - 2;
        const int k0 = first + 1;
        double* gAp = d.Ap + (size_t)line * tw + k0;
        double* gBp = d.Bp + (size_t)line * tw + k0;
        const int nch = sn / RW + 1;
        double ap = 0, bp = 0, xs = 0;
        for (int c = 0; c < nch; ++c) {
            const int rb = RW * c;
            const int re = (rb + RW - 1 < sn) ? rb + RW - 1 : sn;
            for (int r = rb + lane; r <= re; r += 64) {
                const int k = k0 + r;
                const int i = isJ ? k : line, j = isJ ? line : k;
                FsRow w = fs_row<isJ>(d, t, s_start, ketdinh, i, j, first, last, br1, br2);
                sA[r - rb] = w.A; sB[r - rb] = w.B; sC[r - rb] = w.C; sD[r - rb] = w.D;
            }
            __syncthreads();
            if (lane == 0) {
                int q = 0;
                if (rb == 0) {
                    if (sn == 0) {
                        xs = sD[0] / sB[0];
                    } else {
                        ap = -sC[0] / sB[0];
                        bp = sD[0] / sB[0];
                        sA[0] = ap; sB[0] = bp;
                    }
                    q = 1;
                }
                const int qmid = ((re < sn - 1) ? re : sn - 1) - rb;
#pragma unroll 4
                for (; q <= qmid; ++q) {
                    double A = sA[q], B = sB[q], C = sC[q], D = sD[q];
                    double e = A * ap + B;
                    double nap = -C / e;
                    double nbp = (D - (A * bp)) / e;
                    ap = nap;
                    bp = nbp;
                    sA[q] = ap; sB[q] = bp;
                }
                if (re == sn && sn > 0) {
                    double A = sA[sn - rb], B = sB[sn - rb], D = sD[sn - rb];
                    xs = (D - (A * bp)) / (B + (A * ap));
                }
            }
            __syncthreads();
            if (c + 1 < nch)
                for (int q = lane; q <= re - rb; q += 64) { gAp[rb + q] = sA[q]; gBp[rb + q] = sB[q]; }
        }
        for (int c = nch - 1; c >= 0; --c) {
            const int rb = RW * c;
            const int re = (rb + RW - 1 < sn) ? rb + RW - 1 : sn;
            if (c + 1 < nch) {
                __syncthreads();
                for (int q = lane; q <= re - rb; q += 64) { sA[q] = gAp[rb + q]; sB[q] = gBp[rb + q]; }
                __syncthreads();
            }
            if (lane == 0) {
                int q = re - rb;
                if (c == nch - 1) { sD[q] = xs; --q; }
#pragma unroll 4
                for (; q >= 0; --q) {
                    xs = sB[q] + (sA[q] * xs);
                    sD[q] = xs;
                }
            }
            __syncthreads();
            for (int q = lane; q <= re - rb; q += 64) {
                double v = sD[q];
                if (v < 0) v = d.P.NDnen;
                d.tFS[at(k0 + rb + q)] = v;
                if (rb + q == 0) sV[0] = v;
                if (rb + q == sn) sV[1] = v;
            }
        }
        __syncthreads();
        if (lane == 0) {
            const double* tqq = isJ ? d.t_u : d.t_v;
            if ((br1) || (tqq[at(first)] == 0)) d.tFS[at(first)] = sV[0];
            else d.tFS[at(first)] = d.FS[at(first)];
            if ((br2) || (tqq[at(last)] == 0)) d.tFS[at(last)] = sV[1];
            else d.tFS[at(last)] = d.FS[at(last)];
        }
        __syncthreads();
    }
}

/* k_fs_run with the speculative parallel Thomas of hd_thomas.h: rows of a
 * run are assembled in chunks of 256 (four per lane; 8 KB of LDS per
 * workgroup, so that about four workgroups per SIMD fit where a batch has
 * many more runs than the chip has waves), the forward sweep and
 * the back substitution run on all 64 lanes with exact verification, so the
 * bits are those of the serial solve (tridiagSolver with jump 1,
 * UVZSolver_multithread.cu:203-262, via the FS rows of Sediment_Transport.cu:
 * 62-338).
 * One wave per run leaves a SIMD with a wave or two, which issue an
 * instruction every 5 to 7 cycles: the rows' instruction count bounds it.
 * The rows' loads are issued together (the next round's before this one is
 * evaluated), powers of case constants come from the device view, and the
 * rows take the fast form unless a lane's values leave its range: 25-27 us
 * per launch with the plain rows, 18 us with these, on a 980 x 1048 river
 * grid of about 2000 runs. */
template <bool isJ>
__global__ void __launch_bounds__(64) k_fs_spec(const HdDev* __restrict__ dv, double s_start, int ketdinh)
{
    const HdDevG& d = dev_view(dv);
    constexpr int RW = 256;
    /* rows at SpecMap positions (factors replace C / D, x replaces A); the
     * run's first row (0) and last (sn), which the sweeps leave out, at the
     * last two words */
    constexpr int kW = hd_spec::spec_words(RW), kRow0 = kW - 2, kRowN = kW - 1;
    __shared__ double sA[kW], sB[kW], sC[kW], sD[kW];
    const int N = d.N, M = d.M, W = d.W;
    const int lane = threadIdx.x;
    const int tw = 2 * (N > M ? N : M) + 4;
    const int lmax = isJ ? M - 1 : N - 1;
    const int cap = (isJ ? M + 3 : N + 3) * d.SL;
    const int cnt = d.run_cnt[isJ ? 0 : 1] < cap ? d.run_cnt[isJ ? 0 : 1] : cap;
    const int4* runs = isJ ? d.runs_u : d.runs_v;
    const bool src = !(d.tdev[0] < s_start);
    const FsConst K = fs_const(d);
    const RunSlice sl = run_slice(cnt);
    for (int ri = sl.start; ri < sl.end; ri += sl.step) {
        const int4 rn = runs[ri];
        const int line = __builtin_amdgcn_readfirstlane(rn.x), first = __builtin_amdgcn_readfirstlane(rn.y),
                  last = __builtin_amdgcn_readfirstlane(rn.z);
        if (line < 3 || line > lmax || last < first + 2) continue;
        auto at = [&](int k) -> size_t { return isJ ? (size_t)k * W + line : (size_t)line * W + k; };
        const int sn = last - first - 2;
        const int k0 = first + 1;
        const unsigned step = isJ ? 8u * W : 8u;
        auto base = [&](int k) -> long { return isJ ? (long)k * W + line : (long)line * W + k; };
        /* the cells of rows ra .. (64 of them, at most up to row re) */
        auto load = [&](int ra, int re) {
            return fs_load_off<isJ>(d, ketdinh, base(k0 + ra), base(k0 + ra - 1),
                                    (unsigned)(lane < re - ra ? lane : re - ra) * step);
        };
        FsRaw raw = load(0, sn < RW ? sn : RW - 1);
        bool br1, br2;
        wall_flags2(d, isJ, line, first, last, br1, br2);
        const FsEnds E = fs_ends<isJ>(d, line, first, last, br1, br2);
        double* gAp = d.Ap + (size_t)line * tw + k0;
        double* gBp = d.Bp + (size_t)line * tw + k0;
        const int nch = sn / RW + 1;
        double ap = 0, bp = 0, xs = 0;
        double ap0 = 0, bp0 = 0; /* row 0's factors */
        /* rows of chunk c that the sweeps take: rb .. rb + n - 1 */
        auto chunk_rows = [&](int c, int& rb, int& n) {
            const int re = RW * (c + 1) - 1 < sn - 1 ? RW * (c + 1) - 1 : sn - 1;
            rb = c == 0 ? 1 : RW * c;
            n = re - rb + 1;
        };
        for (int c = 0; c < nch; ++c) {
            int rb, n;
            chunk_rows(c, rb, n);
            const hd_spec::SpecMap sm = hd_spec::spec_map(n);
            const int ra = RW * c, re = ra + RW - 1 < sn ? ra + RW - 1 : sn; /* assembled rows */
            if (c > 0) raw = load(ra, re);
            for (int r0 = ra; r0 <= re; r0 += 64) {
                const int r = r0 + lane;
                FsRaw x = raw;
                if (r0 + 64 <= re) raw = load(r0 + 64, re);
                fs_before<isJ>(x);
                FsGuard G;
                FsRow w = fs_eval<isJ, true>(d, K, x, E, src, ketdinh, r == 0, r == sn, G);
                if (__any(!(K.ok && G.ok()))) {
                    FsGuard G2;
                    w = fs_eval<isJ, false>(d, K, x, E, src, ketdinh, r == 0, r == sn, G2);
                }
                if (r <= re) {
                    const int p = r == 0 ? kRow0 : (r == sn ? kRowN : sm.pos(r - rb));
                    sA[p] = w.A; sB[p] = w.B; sC[p] = w.C; sD[p] = w.D;
                }
            }
            __syncthreads();
            if (c == 0) {
                if (sn == 0) {
                    xs = sD[kRow0] / sB[kRow0];
                } else {
                    ap0 = ap = -sC[kRow0] / sB[kRow0];
                    bp0 = bp = sD[kRow0] / sB[kRow0];
                }
            }
            hd_spec::spec_forward<2>(sA, sB, sC, sD, sm, n, ap, bp);
            if (c == nch - 1 && sn > 0) {
                const double A = sA[kRowN], B = sB[kRowN], D = sD[kRowN];
                xs = (D - (A * bp)) / (B + (A * ap));
            }
            if (c + 1 < nch) {
                for (int r = lane; r < n; r += 64) {
                    gAp[rb + r] = sC[sm.pos(r)];
                    gBp[rb + r] = sD[sm.pos(r)];
                }
                __syncthreads();
            }
        }
        double xc = xs;
        for (int c = nch - 1; c >= 0; --c) {
            int rb, n;
            chunk_rows(c, rb, n);
            const hd_spec::SpecMap sm = hd_spec::spec_map(n);
            if (c + 1 < nch) {
                __syncthreads();
                for (int r = lane; r < n; r += 64) {
                    sC[sm.pos(r)] = gAp[rb + r];
                    sD[sm.pos(r)] = gBp[rb + r];
                }
                __syncthreads();
            }
            xc = hd_spec::spec_backward<2>(sC, sD, sA, sm, n, xc);
            if (c == 0 && sn > 0) xc = bp0 + (ap0 * xc);
            const int r0 = c == 0 ? 0 : rb, r1 = c == nch - 1 ? sn : rb + n - 1;
            for (int r = r0 + lane; r <= r1; r += 64) {
                double v = r == sn ? xs : (r == 0 ? xc : sA[sm.pos(r - rb)]);
                if (v < 0) v = d.P.NDnen;
                st_off(d.tFS, base(k0 + r0), (unsigned)(r - r0) * step, v);
            }
        }
        /* the end cells: the neighbour's value, or their own */
        if (lane == 0) {
            double v1 = sn == 0 ? xs : xc, v2 = xs;
            if (v1 < 0) v1 = d.P.NDnen;
            if (v2 < 0) v2 = d.P.NDnen;
            d.tFS[at(first)] = E.w1 ? v1 : E.f1;
            d.tFS[at(last)] = E.c2 ? v2 : E.f2;
        }
        __syncthreads();
    }
}

/* Update_FS, Sediment_Transport.cu:620-629. */
__global__ void __launch_bounds__(256) k_update_fs(const HdDev* __restrict__ dv, int tiled)
{
    const HdDevG& d = dev_view(dv);
    int j, i;
    if (tiled) {
        if (!tile_cell(d, i, j)) return;
        if (i < 1 || j < 1) return;
    } else {
        j = blockIdx.x * blockDim.x + threadIdx.x + 1;
        i = blockIdx.y + 1;
    }
    if (i > d.N || j > d.M) return;
    d.FS[i * d.W + j] = d.tFS[i * d.W + j];
}

/* Calculate_Qb, Sediment_Transport.cu:341-414 (qb_mode REFERENCE keeps the
 * `!VTH` test as written, FIXED uses VTH != 0; corner copies braced).  Two
 * fluxes share one power; the other two are of case constants and come from
 * the device view: 5.0 us on a 980 x 1048 river grid, 10.7 with eight
 * powers per cell.  With `update` (tiles only) it also does Update_FS of the
 * half-step before, whose values it does not read: a launch of 5 us less. */
__global__ void __launch_bounds__(256) k_calc_qb(const HdDev* __restrict__ dv, int qb_mode, int tiled, int update)
{
    const HdDevG& d = dev_view(dv);
    int j, i;
    if (tiled) {
        if (!tile_cell(d, i, j)) return;
        if (update && i >= 1 && j >= 1 && i <= d.N && j <= d.M) d.FS[i * d.W + j] = d.tFS[i * d.W + j];
        if (i < 2 || j < 2) return;
    } else {
        j = blockIdx.x * blockDim.x + threadIdx.x + 2;
        i = blockIdx.y + 2;
    }
    int N = d.N, M = d.M, W = d.W;
    if (i > N || j > M) return;
    const hd_params& P = d.P;
    double* Qbx = d.Qbx;
    double* Qby = d.Qby;
    int pos = i * W + j;
    double Tob, Toee = P.Toe, Tx = 0;
    /* one round of loads */
    const double vth = d.VTH[pos], fw = d.Fw[pos], hm = d.H_moi[pos];
    const double us = d.t_u[pos] + d.t_u[pos - W], vs = d.t_v[pos] + d.t_v[pos - 1];
    const int kh = d.khouot[pos];
    const bool sel = (qb_mode == HD_QB_REFERENCE) ? (!vth) : (vth != 0);
    double qx = 0, qy = 0;
    if (sel && (kh == 0)) {
        Tob = P.ro * fw * (vth * vth);
        if (hm > P.ghtoe) Toee = P.Toe * (1 + P.hstoe * ((hm - P.ghtoe)));
        if (Tob > Toee) Tx = Tob / Toee - 1;
        /* 0.053 ((Sx - 1) g)^0.5 dm^1.5 Tx^2.1 Dxr^-0.3, the factors of both directions */
        const double c = d.Qb_c * hd_pow(Tx, 2.1) * d.Dxr_m03;
        qx = c * us * 0.5 / vth;
        qy = c * vs * 0.5 / vth;
    }
    Qbx[pos] = qx;
    Qby[pos] = qy;
    if (i == 2) { Qbx[pos - W] = qx; Qby[pos - W] = qy; }
    if (i == N) { Qbx[pos + W] = qx; Qby[pos + W] = qy; }
    if (j == 2) {
        Qbx[pos - 1] = qx; Qby[pos - 1] = qy;
        if (i == 2) { Qbx[1 * W + 1] = qx; Qby[1 * W + 1] = qy; }
        if (i == N) { Qbx[(N + 1) * W + 1] = qx; Qby[(N + 1) * W + 1] = qy; }
    }
    if (j == M) {
        Qbx[pos + 1] = qx; Qby[pos + 1] = qy;
        if (i == 2) { Qbx[1 * W + M + 1] = qx; Qby[1 * W + M + 1] = qy; }
        if (i == N) { Qbx[(N + 1) * W + M + 1] = qx; Qby[(N + 1) * W + M + 1] = qy; }
    }
}

/* _bed_load via BedLoad, Sediment_Transport.cu:416-506 / 630-639: rows
 * [sidx, eidx-1], cells of row runs with last - first >= 2 (t_u[pos > 0]
 * reads t_u[1], as written).  The loads do not wait for the tests that
 * choose among them, and the source term takes the rows' fast form: 7.7 us
 * on a 980 x 1048 river grid, 12 without. */
__global__ void __launch_bounds__(256) k_bedload(const HdDev* __restrict__ dv, int ketdinh, int slo, int eoff, int tiled)
{
    const HdDevG& d = dev_view(dv);
    const int sidx = slo, eidx = d.N - eoff;
    int N = d.N, M = d.M, W = d.W, SL = d.SL;
    int i, j;
    int first = 0, last = 0;
    bool found = false;
    if (tiled) { /* run cells lie in the active tiles; the row's table is wave-uniform */
        if (!tile_cell(d, i, j)) return;
        if (i < sidx || i >= eidx || j < 2 || j > M) return;
        const int moc = min(d.moci[i], SL);
        for (int s = 0; s < moc; ++s) {
            const int a = d.daui[i * SL + s], b = d.cuoii[i * SL + s];
            if (a <= j && j <= b) { first = a; last = b; found = true; break; }
        }
    } else {
        __shared__ int s_moc;
        __shared__ int s_dau[24], s_cuoi[24];
        i = sidx + blockIdx.y;
        if (i >= eidx) return;
        if (threadIdx.x == 0) s_moc = min(d.moci[i], SL);
        __syncthreads();
        if (threadIdx.x < s_moc) { s_dau[threadIdx.x] = d.daui[i * SL + threadIdx.x]; s_cuoi[threadIdx.x] = d.cuoii[i * SL + threadIdx.x]; }
        __syncthreads();
        j = blockIdx.x * blockDim.x + threadIdx.x + 2;
        if (j > M) return;
        for (int s = 0; s < s_moc; ++s)
            if (s_dau[s] <= j && j <= s_cuoi[s]) { first = s_dau[s]; last = s_cuoi[s]; found = true; break; }
    }
    if (!found || last - first < 2) return;
    const hd_params& P = d.P;
    const int pos = i * W + j;
    /* one round of loads: the cell, and its neighbours up to two away */
    const double *FS = d.FS, *Qbx = d.Qbx, *Qby = d.Qby;
    const int* kh = d.khouot;
    const double x0 = Qbx[pos], xp1 = Qbx[pos + W], xp2 = Qbx[pos + 2 * W], xm1 = Qbx[pos - W], xm2 = Qbx[pos - 2 * W];
    const double y0 = Qby[pos], yp1 = Qby[pos + 1], yp2 = Qby[pos + 2], ym1 = Qby[pos - 1], ym2 = Qby[pos - 2];
    const bool kxp1 = kh[pos + W] == 1, kxp2 = kh[pos + 2 * W] == 1, kxm1 = kh[pos - W] == 1, kxm2 = kh[pos - 2 * W] == 1;
    const bool kyp1 = kh[pos + 1] == 1, kyp2 = kh[pos + 2] == 1, kym1 = kh[pos - 1] == 1, kym2 = kh[pos - 2] == 1;
    const double f0 = FS[pos], fxp = FS[pos + W], fxm = FS[pos - W], fyp = FS[pos + 1], fym = FS[pos - 1];
    const double hu0 = d.Htdu[pos], hum = d.Htdu[pos - W], hv0 = d.Htdv[pos], hvm = d.Htdv[pos - 1];
    const double kx0 = d.Kx[pos], kxm = d.Kx[pos - W], ky0 = d.Ky[pos], kym = d.Ky[pos - 1];
    const double u0 = d.t_u[pos], u1 = d.t_u[1], v0 = d.t_v[pos];
    const double hm = d.H_moi[pos], vth = d.VTH[pos], fw = d.Fw[pos], dH = d.dH[pos];
    /* the bed-load gradients: one-sided at a wall and only for flow away
     * from it, else central */
    double p = kxm1 ? -3 * x0 + 4 * xp1 - xp2 : kxp1 ? 3 * x0 - 4 * xm1 + xm2 : xp1 - xm1;
    const bool onx = kxm1 ? u0 < 0 : (kxp1 ? u1 != 0 : true);
    p = onx ? p / P.dX2 : 0.0;
    double q = kym1 ? -3 * y0 + 4 * yp1 - yp2 : kyp1 ? 3 * y0 - 4 * ym1 + ym2 : yp1 - ym1;
    const bool ony = kym1 ? v0 < 0 : (kyp1 ? v0 > 0 : true);
    q = ony ? q / P.dY2 : 0.0;
    double tH = p + q;
    p = fxp - f0;
    if ((kxp2 || kxm1) && (i < N)) p = 0;
    q = f0 - fxm;
    if ((i > 2) && (kxm2 || kxp1)) q = 0;
    p = 1 / P.dXbp * (hu0 * kx0 * p - hum * kxm * q);
    tH = tH + p;
    p = fyp - f0;
    if (((last < M) && (kym1 || kyp2)) || (last == M && kym1)) p = 0;
    q = f0 - fym;
    if (((first > 2) && (kym2 || kyp1)) || (first == 2 && kyp1)) q = 0;
    p = 1 / (P.dYbp) * (hv0 * ky0 * p - hvm * kym * q);
    tH = tH + p;
    const FsConst K = fs_const(d);
    FsGuard G;
    double Zf;
    double S = fs_source<true>(d, K, ketdinh, 0.0, hm, f0, vth, fw, Zf, G);
    if (__any(!(K.ok && G.ok() && hd_div::finite(S)))) S = fs_source<false>(d, K, ketdinh, 0.0, hm, f0, vth, fw, Zf, G);
    d.dH[pos] = dH + P.dT / (1 - P.Dorong) * (S + tH);
}

} // namespace

static inline dim3 tile_grid(const HdBatch& b, int ntiles) { return dim3((ntiles + 3) / 4, 1, b.n); }

void hd_launch_vth_hesok(const HdBatch& b, int ntiles, int bnd, hipStream_t s)
{
    if (ntiles > 0) {
        dim3 g = tile_grid(b, ntiles);
        g.x += bnd;
        hipLaunchKernelGGL(k_vth_hesok, g, dim3(256), 0, s, b.dv, 1, bnd);
        return;
    }
    dim3 g2((b.M + 1 + 255) / 256, b.N + 1, b.n);
    hipLaunchKernelGGL(k_vth_hesok, g2, dim3(256), 0, s, b.dv, 0, 0);
}

void hd_launch_fs_coef(const HdBatch& b, int which, double s_start, int ketdinh, hipStream_t s)
{
    dim3 blk(64, 4);
    dim3 grd((b.M + 3 + 63) / 64, (b.N + 3 + 15) / 16, b.n);
    if (which == 0) hipLaunchKernelGGL(k_fs_coef<true>, grd, blk, 0, s, b.dv, s_start, ketdinh);
    else hipLaunchKernelGGL(k_fs_coef<false>, grd, blk, 0, s, b.dv, s_start, ketdinh);
}

void hd_launch_fs_solve(const HdBatch& b, int which, hipStream_t s)
{
    int nl = (which == 0 ? b.M : b.N) - 3;
    if (nl <= 0) return;
    if (which == 0) hipLaunchKernelGGL(k_fs_solve<true>, dim3((nl + 63) / 64, 1, b.n), dim3(64), 0, s, b.dv);
    else hipLaunchKernelGGL(k_fs_solve<false>, dim3((nl + 63) / 64, 1, b.n), dim3(64), 0, s, b.dv);
}

void hd_launch_update_fs(const HdBatch& b, int ntiles, hipStream_t s)
{
    if (ntiles > 0) {
        hipLaunchKernelGGL(k_update_fs, tile_grid(b, ntiles), dim3(256), 0, s, b.dv, 1);
        return;
    }
    hipLaunchKernelGGL(k_update_fs, dim3((b.M + 255) / 256, b.N, b.n), dim3(256), 0, s, b.dv, 0);
}

void hd_launch_calc_qb(const HdBatch& b, int qb_mode, int ntiles, int update, hipStream_t s)
{
    if (ntiles > 0) {
        hipLaunchKernelGGL(k_calc_qb, tile_grid(b, ntiles), dim3(256), 0, s, b.dv, qb_mode, 1, update);
        return;
    }
    hipLaunchKernelGGL(k_calc_qb, dim3((b.M - 1 + 255) / 256, b.N - 1, b.n), dim3(256), 0, s, b.dv, qb_mode, 0, 0);
}

void hd_launch_bedload(const HdBatch& b, int ketdinh, int slo, int eoff, int ntiles, hipStream_t s)
{
    if (ntiles > 0) {
        hipLaunchKernelGGL(k_bedload, tile_grid(b, ntiles), dim3(256), 0, s, b.dv, ketdinh, slo, eoff, 1);
        return;
    }
    int nr = b.N - eoff - slo;
    if (nr > 0)
        hipLaunchKernelGGL(k_bedload, dim3((b.M - 1 + 255) / 256, nr, b.n), dim3(256), 0, s, b.dv, ketdinh, slo, eoff, 0);
}

void hd_launch_fs_line(const HdBatch& b, int which, double s_start, int ketdinh, hipStream_t s)
{
    int nl = (which == 0 ? b.M : b.N) - 3;
    if (nl <= 0) return;
    if (which == 0) hipLaunchKernelGGL(k_fs_line<true>, dim3(nl, 1, b.n), dim3(64), 0, s, b.dv, s_start, ketdinh);
    else hipLaunchKernelGGL(k_fs_line<false>, dim3(nl, 1, b.n), dim3(64), 0, s, b.dv, s_start, ketdinh);
}

void hd_launch_fs_run(const HdBatch& b, int which, double s_start, int ketdinh, int nblocks, int spec, hipStream_t s)
{
    dim3 g(nblocks, 1, b.n);
    if (spec) {
        if (which == 0) hipLaunchKernelGGL(k_fs_spec<true>, g, dim3(64), 0, s, b.dv, s_start, ketdinh);
        else hipLaunchKernelGGL(k_fs_spec<false>, g, dim3(64), 0, s, b.dv, s_start, ketdinh);
    } else {
        if (which == 0) hipLaunchKernelGGL(k_fs_run<true>, g, dim3(64), 0, s, b.dv, s_start, ketdinh);
        else hipLaunchKernelGGL(k_fs_run<false>, g, dim3(64), 0, s, b.dv, s_start, ketdinh);
    }
}
