/*
 * hd_edges.h -- the boundary values of a half-step from the hourly series
 * (Update_Boundary_Value, support_funcs.cu:622-668), for the launches that
 * write them with a workgroup of their own: k_boundary, and k_vth_hesok on a
 * frozen flow.
 */
#ifndef HD_EDGES_H
#define HD_EDGES_H

#include "hd_internal.h"

/* Edge e (up, down, left, right) over its line's first wet run, the only one
 * the reference updates (support_funcs.cu:558), by STRIDE threads (lt: the
 * thread among them), U cells a thread in one round of loads.  All threads of
 * the workgroup call it, between them with every e; the half-step's time
 * t = t_prev + dT/2 is advanced here.  A thread reads the device time and its
 * edge's tables in one round, the series values and the cells' weights follow
 * in a second. */
template <int STRIDE, int U>
__device__ __forceinline__ void boundary_series(const HdDevG& d, int e, int lt)
{
    double* tdev = d.tdev;
    const double t = tdev[0] + d.P.dT * 0.5;
    const int N = d.N, M = d.M, W = d.W, SL = d.SL, TT = d.total_time;
    const int imax = M > N ? M : N;
    const bool isU = e >= 2;
    const int* moc = isU ? d.moci : d.mocj;
    const int* dau = isU ? d.daui : d.dauj;
    const int* cuoi = isU ? d.cuoii : d.cuoij;
    const int location = e == 0 ? M : (e == 3 ? N : 2);
    const int loc_ext = e == 0 ? M + 1 : (e == 3 ? N + 1 : 1);
    const int mc = moc[location], a = dau[location * SL], b = cuoi[location * SL];
    const int bt0 = d.boundary_type[e * SL];
    const double hmax = d.hmax[e];
    /* row-edge coverage of the corner cells (rows 2 and N) of the column edges */
    const int m2 = d.moci[2], a2 = d.daui[2 * SL], b2 = d.cuoii[2 * SL], rbt2 = d.boundary_type[2 * SL];
    const int mN = d.moci[N], aN = d.daui[N * SL], bN = d.cuoii[N * SL], rbt3 = d.boundary_type[3 * SL];
    __syncthreads(); /* every thread has read the old time */
    if (threadIdx.x == 0) tdev[0] = t;
    const int t1 = (int)(t / 3600);
    const double t2 = (t - (3600.0 * t1)) / 3600.0;
    if (t1 < 0 || t1 + 1 >= TT || t1 + 1 >= d.series_len) {
        if (threadIdx.x == 0) d.flags[1] = 1;
        return;
    }
    if (mc <= 0) return;
    const double* bc = e == 0 ? d.bc_up : e == 1 ? d.bc_down : e == 2 ? d.bc_left : d.bc_right;
    const double* CCs = e == 0 ? d.CC_u : e == 1 ? d.CC_d : e == 2 ? d.CC_l : d.CC_r;
    const double* hi = d.hi + (e == 0 ? 0 : e == 1 ? (N + 3) : e == 2 ? 2 * (N + 3) : 2 * (N + 3) + (M + 3));
    double* barr = e == 0 ? d.vbt : e == 1 ? d.vbd : e == 2 ? d.ubt : d.ubp;
    const int last = b < imax ? b : imax;
    for (int i0 = (a > 2 ? a : 2) + lt; i0 <= last; i0 += STRIDE * U) {
        /* Boundary_value + FS_boundary, support_funcs.cu:544-617, segment 0 */
        const double b0 = bc[t1], b1 = bc[t1 + 1];
        const double c0 = CCs[t1], c1 = CCs[t1 + 1];
        double hw[U], hbd[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * STRIDE <= last ? i0 + u * STRIDE : last;
            const int fi = isU ? location : i, fj = isU ? i : location;
            hw[u] = hi[i];
            hbd[u] = d.htaiz_bd[fi * W + fj];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * STRIDE;
            if (i > last) break;
            const int fi = isU ? location : i, fj = isU ? i : location;
            /* a column edge (0, 1) leaves its cell of row 2 / N to the row edge
             * (2 / 3) that writes the same field there: in the reference's edge
             * order the later edge wins */
            bool yield = false;
            if (!isU && (i == 2 || i == N)) {
                const bool covers = (i == 2) ? (m2 > 0 && a2 <= location && location <= b2)
                                             : (mN > 0 && aN <= location && location <= bN);
                const int rb0 = (i == 2) ? rbt2 : rbt3;
                yield = covers && ((rb0 == 2) == (bt0 == 2));
            }
            const double bv = b0 * (1.0 - t2) + b1 * t2;
            if (bt0 == 2) {
                barr[i] = bv * hw[u];
            } else if (isU) {
                d.t_z[location * W + i] = bv;
                d.t_z[loc_ext * W + i] = bv;
            } else {
                if (!yield) d.t_z[i * W + location] = bv;
                d.t_z[i * W + loc_ext] = bv;
            }
            if (bt0 != 2 || yield) continue;
            const double cv = c0 * (1.0 - t2) + c1 * t2;
            d.FS[fi * W + fj] = cv * hbd[u] * hmax;
        }
    }
}

#endif
