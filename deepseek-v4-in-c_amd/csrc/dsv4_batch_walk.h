/* SPDX-License-Identifier: Apache-2.0 */
/* dsv4_batch_walk.h - the order in which a wave of k_batch_mf
 * (dsv4_batch_mf.hip) walks its part of a row: integers only, so that the
 * host can check every index it gives. */
#ifndef DSV4_BATCH_WALK_H
#define DSV4_BATCH_WALK_H

#ifdef __HIPCC__
#define DSV4_HD __host__ __device__ __forceinline__
#else
#define DSV4_HD inline
#endif

/* The wave's slots j0 .. j0 + L - 1 in groups of four; group u at pass n is
 * the chunks j0 + 4 u + n tc .. + 3. A step is a (u, n) whose first chunk
 * lies in the row of ch chunks, n fastest. */
struct MfWalk {
    int u = 0, n = 0, c;                       /* the step, its first chunk */

    DSV4_HD explicit MfWalk(int j0) : c(j0) {}
    DSV4_HD void next(int j0, int tc, int ch)
    {
        n++;
        c += tc;
        if (c >= ch) {
            u++;
            n = 0;
            c = j0 + 4 * u;
        }
    }
    /* its place in the table of `groups` = (L / 4) nch entries. A wave reads
     * the operands of one step more than it has; after a wave whose last
     * group lies in the row, that one is past the table: it reads the last
     * entry again. */
    DSV4_HD int entry(int nch, int groups) const
    {
        const int i = u * nch + n;
        return i < groups ? i : groups - 1;
    }
};

/* The steps of such a wave; nch = ceil(ch / tc), so only the last pass of a
 * group in the row can lie outside it. No loop: the first copies wait for
 * this (1024x4096 BF16 at 48 tokens 10.81 us with a loop over the groups). */
DSV4_HD int mf_steps(int j0, int L, int tc, int ch, int nch)
{
    const int groups = L >> 2, rest = ch - (nch - 1) * tc;     /* the last pass's chunks */
    const int in_row = j0 < ch ? (ch - j0 + 3) >> 2 : 0, last = j0 < rest ? (rest - j0 + 3) >> 2 : 0;
    return (groups < in_row ? groups : in_row) * (nch - 1) + (groups < last ? groups : last);
}

#endif
