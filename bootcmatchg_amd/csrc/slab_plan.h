/*
 * slab_plan.h - how several sweeps of an interleaved block split into
 * workgroups (k_il_slab of kernels_multi.hip). No HIP.
 */
#pragma once

namespace bcmg {

/* lanes of a slab's workgroup, which holds four cells a lane at most */
constexpr int SLAB_BS = 1024;

/* The slab of `sweeps` sweeps: the rows a workgroup stores and its cells per
   lane (0: does not fit). */
struct IlSlab {
    int L = 0, rpt = 0;
    double us = 0;
};

/* Predicted time: a launch, the loads and the store cost about 4.5 us, a sweep
   of the cells 0.45 us per cell of a lane and round of workgroups (one a CU);
   a sweep of its own 3 us and its bytes at 8 TB/s. */
inline IlSlab il_slab_fit(int n, int band, int gpr, int sweeps)
{
    IlSlab best;
    const long long halo = (long long)band * sweeps; /* any band: an offset of an int */
    for (int L = 16; L <= 512; L *= 2) {
        const long long cells = (L + 2 * halo) * gpr;
        if (cells > 4 * SLAB_BS) break;
        const int rpt = (int)((cells + SLAB_BS - 1) / SLAB_BS);
        const int rounds = (int)((n + 256ll * L - 1) / (256 * L));
        const double us = 2.5 + rounds * (2.0 + sweeps * 0.45 * rpt);
        if (best.rpt == 0 || us < best.us) best = IlSlab{L, rpt, us};
    }
    return best;
}

} // namespace bcmg
