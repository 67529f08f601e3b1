// The small end of the V-cycle as one dense operator (see lal_coarse.hip).
#pragma once

#include "lal_internal.h"

namespace lal
{
    // Rows of the largest level whose cycle is kept as a dense operator: 8 MB,
    // which the eight L2s hold beside the level above.  Up to here it replaces
    // four or more launches of 3 to 4 us (an iteration of PCG on 128^2 Poisson,
    // where the level has 496 rows, 69 -> 52 us; on 64^3 with 1000 rows
    // 208 -> 181 us with the hierarchy's build) for three launches a level in the
    // setup, which the packing of the levels into an LDS image cost before.
    // The operator grows with the square, its construction faster; the next
    // larger levels of the grids measured (3,500 to 4,000 rows) would read 100 MB.
    constexpr int CYCLE_ROWS = 1024;

    // One level as the construction reads it (FP64): A and 1/a_ii, the
    // restriction R (mc x m) and Q = P - D^-1 A P (m x mc).
    struct cycle_level
    {
        int           m, mc;
        const int *   arp, *aci;
        const double *av, *dinv;
        const int *   rrp, *rci;
        const double* rv;
        const int *   qrp, *qci;
        const double* qv;
    };

    // Leading dimension of a level's operator.
    __host__ __device__ inline int cycle_ld(int m)
    {
        return (m + 1) & ~1;
    }

    // M (m rows of cycle_ld(m)): the level's V-cycle from zero with one pre- and
    // one post-sweep, given the next level's operator Mc (mc rows of ldc) or, for
    // a 1x1 coarsest level, its entry a11.  S and U: mc x cycle_ld(m) scratch.
    int cycle_matrix(lal_context* c, const cycle_level& L, const double* Mc, int ldc,
                     const double* a11, double* S, double* U, double* M);

    // x = M b
    template <typename T>
    int cycle_apply(lal_context* c, int m, const double* M, const T* b, T* x);
}
