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

} // namespace bcmg
