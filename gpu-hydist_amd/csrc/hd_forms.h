/*
 * hd_forms.h -- which form of a computation a lane, a line or a batch takes,
 * as plain functions of numbers: the kernels and the host share them, and so
 * does a test that compiles them for the host.
 */
#ifndef HD_FORMS_H
#define HD_FORMS_H

#if defined(__HIP__)
#define HD_FORM __host__ __device__ static inline
#else
#define HD_FORM static inline
#endif

/* The momentum row of cell k of run [first, last] as lane `lane` of a round
 * of 63 cells assembles it: whether it has one, and whether the terms of the
 * face behind and of the face ahead enter it (not at a wall, br1 / br2, and
 * not in a run of two cells).  Lane 63 holds the next round's first cell for
 * its continuity coefficients alone: it has no lane after it to take the face
 * ahead's from, and its row is that round's. */
struct HdCellUse {
    bool row, behind, ahead;
};
HD_FORM HdCellUse hd_cell_use(int lane, int k, int first, int last, bool br1, bool br2)
{
    HdCellUse u;
    const bool inner = last - 1 > first;
    u.row = lane < 63 && k < last;
    u.behind = inner && !(br1 && k == first);
    u.ahead = inner && !(br2 && k == last - 1);
    return u;
}

/* The wetting pass of a line with n recorded candidates, of which the list
 * holds `most`; dependent: candidates near each other, or a cascade that
 * leaves its window.  mode (HYDIST_WETTING): 1 the replay for every line, 2
 * the scan. */
enum { HD_WET_AT_ONCE, HD_WET_REPLAY, HD_WET_SCAN };
HD_FORM int hd_wet_form(int mode, int n, int most, bool dependent)
{
    if (n > most || mode == 2) return HD_WET_SCAN;
    return mode == 1 || dependent ? HD_WET_REPLAY : HD_WET_AT_ONCE;
}

#endif
