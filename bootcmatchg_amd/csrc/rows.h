/*
 * rows.h - which row a group of lanes takes, and how many workgroups rows of
 * such groups need. No HIP: the functions run on the host and the device.
 */
#pragma once

namespace bcmg {

/* lanes of a workgroup of the row kernels */
constexpr int ROW_BS = 256;

/* The row of a thread where G lanes (a power of two up to ROW_BS) take one:
   formed from the block, since (block ROW_BS + thread) passes 2^31 where rows x
   G does, at 1.1e9 entries. */
constexpr int group_row(unsigned block, unsigned thread, int G)
{
    return (int)(block * (unsigned)(ROW_BS / G) + thread / (unsigned)G);
}

/* The rows of [0, n) whose neighbours at offsets lo to hi lie in it too: from
   `first` on and before `last`. A block of rows from r0 on is inside then when
   r0 >= first and r0 <= last - rows; r0 + hi would pass 2^31 from 2^30 rows on. */
struct InnerRows {
    int first, last;
    constexpr bool holds(int r0, int rows) const { return r0 >= first && r0 <= last - rows; }
};
constexpr InnerRows inner_rows(int n, int lo, int hi)
{
    return InnerRows{lo < 0 ? -lo : 0, n - (hi > 0 ? hi : 0)};
}

/* Workgroups for n rows of G lanes. A launch takes less than 2^32 lanes, which
   a wavefront a row reaches at 2^26 rows: the grid is capped at 2^31 lanes and
   the kernels step by it (row_step). */
constexpr int group_blocks(int n, int G)
{
    const long long rows = ROW_BS / G, b = (n + rows - 1) / rows;
    return (int)(b < (1 << 23) ? b : (1 << 23));
}

/* rows that a whole grid takes at once */
constexpr long long row_step(unsigned blocks, int G)
{
    return (long long)blocks * (ROW_BS / G);
}

} // namespace bcmg
