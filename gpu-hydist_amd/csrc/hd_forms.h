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

/* Whether a batch of nsys tridiagonal systems, `some` of which have `rows`
 * rows together, goes by a lane per system rather than a wave.  A lane takes about 0.75 us per row of
 * the longest system, waves about 4.2 us for every 2048 systems (eight
 * workgroups of 18 KB of LDS on each of 256 CUs): the lane form where the
 * first is less.  Measured, lane against wave form, us: 4 rows x 64 systems
 * 3.4 / 4.2, 8 x 64 4.8 / 4.1, 8 x 2000 5.1 / 6.1, 12 x 2000 6.9 / 6.2, 16 x
 * 2000 11 / 6.1, 24 x 20000 24 / 48, 32 x 20000 32 / 46, 64 x 20000 61 / 53,
 * 64 x 2000 41 / 7.5. */
HD_FORM bool hd_thomas_lanes(int nsys, int some, long long rows) { return (nsys + 2048LL) * some > 384 * rows; }

#endif
