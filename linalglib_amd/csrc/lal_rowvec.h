// Fast (non-exact) CSR kernels.
//
// A 256-lane workgroup owns one row block of the analysis (at most 256 rows,
// at most 2048 nonzeros unless a single row is longer).  The main kernel
// (16-byte aligned column and value arrays) copies the block's column indices
// and values into LDS with 16-byte non-temporal loads, four nonzeros per lane,
// and then lets every row -- one lane, or a group of G lanes with a fixed
// butterfly in blocks of few long rows -- walk its own nonzeros in LDS and
// gather x itself, eight (G = 1) or four gathers in flight per lane.  A gather
// instruction then touches the same stencil offset of consecutive rows.  For
// the rectangular transfer operators (P: 4-7 nonzeros per row, R: their
// transposes) the lanes instead gather x for the consecutive nonzeros they
// loaded and stage the products, which wastes no lanes on short rows.
// Unaligned arrays take the product-staging kernel: lanes gather x for
// consecutive nonzeros and stage a_ij * x_j in LDS before the row sums.
// Column indices and values are read once per call, so they are streamed
// (non-temporal) and x keeps the caches -- except for operators marked `keep`
// (a hierarchy's, as many as share the Infinity Cache), whose ordinary loads
// let them stay there between calls.  The sum order differs from the
// host's sequential fma, so results agree to rounding, deterministically; the
// bit-exact path is the row-block kernel of lal_csrmv.hip.
//
// All level operations are one kernel with different gathers and epilogues:
//   SPMV      y = alpha*(A x) + beta*y
//   RESIDUAL  y = b - A x
//   JACOBI    y = x + (b - A x) * dinv     (= (b - sum_{k!=i} a_ik x_k)/a_ii)
//   JACOBI0   y = b * dinv and r = b - A (b * dinv)  (one sweep from x = 0,
//                                           fused with the residual)
//   RESTRICT  y = A x and r = y * dinv     (restriction that also writes the
//                                           coarse level's first sweep)
//   SMOOTHED  y = b - A x and r = x + y * dinv  (residual, and the sweep that
//                                           uses it)
//   ADD       y = b + A x
//   SPMV_DOT  y = A x, ADD_DOT  y = b + A x, and one partial of <w, y> per row
//             block (PCG's inner products without a pass of their own)
//   STEP_DOT  p' = x + beta p, y = A p' and <p', y>'s partials: PCG's next
//             direction formed by the product that needs it
// dinv holds 1/a_ii, so no division is left in the inner loops.
#pragma once

#include "lal_reduce.h"

namespace lal
{
    enum
    {
        RV_SPMV     = 0,
        RV_RESIDUAL = 1,
        RV_JACOBI   = 2,
        RV_JACOBI0  = 3,
        RV_RESTRICT = 4, // y = A x and r = y * dinv: the coarse right-hand side
                         // and the first Jacobi iterate from zero on it
        RV_SMOOTHED = 5,
        RV_ADD      = 6,
        RV_SPMV_DOT = 7,
        RV_ADD_DOT  = 8,
        RV_STEP_DOT = 9
    };

    // Partials of one reduction at most: a product with more row blocks leaves
    // its inner product to a kernel of its own.  Every block of the next kernel
    // adds the partials up again; with fused products the solver saves a pass
    // over two vectors and a launch (2.6 us each at 16,384 rows, 128^2 Poisson
    // 52 -> 44 us per iteration together with the folded norm).  Up to 4096
    // partials nothing measured is slower than with 512 (PCG on 64^3 16.15 ->
    // 16.05 ms, on 101^3 even); 16384 cost 128^3 in FP32 1.3 %.
    constexpr int PCG_PARTS = 4096;

    // What a product does besides its own rows: the *_DOT modes...
    struct row_dot
    {
        double*     part = nullptr; // one partial of <w, y> per row block
        const void* w    = nullptr; // m entries, FP64 with `wide`, else of the product's type
        bool        wide = false;
        // STEP_DOT: beta = (sum of the gamma_count partials at gamma_part) / *gamma_old,
        // whose numerator also goes to *gamma_new
        const double* gamma_part  = nullptr;
        int           gamma_count = 0;
        const double* gamma_old   = nullptr;
        double*       gamma_new   = nullptr;
    };
    // ... and SMOOTHED, whose last workgroup finishes the reduction before it.
    struct row_extra : row_dot
    {
        post_args post{};
    };

    struct rv_args
    {
        int         m;
        int         nnz;
        int         by_nnz; // gather over consecutive nonzeros (transfer operators)
        const int*  blocks; // analysis row blocks (nb + 1)
        int         nb;
        const int*  rp;
        const int*  ci;
        const void* val;
        const void* x;
        const void* d;
        const void* b;
        void*       y;
        void*       r;
        double      alpha;
        double      beta;
        int         win; // LDS window in entries (lal_csrmv_info::win)
        int         keep = 0; // the matrix may stay in the cache (lal_csrmv_info::keep)
        // 16-bit columns and their per-block bases (lal_csrmv_info::d_c16), or null
        const unsigned short* c16   = nullptr;
        const int*            cbase = nullptr;
        // column lists (lal_csrmv_info::d_list), list_max 0: none
        const unsigned short* lpos     = nullptr;
        const unsigned short* list     = nullptr;
        const int*            lmeta    = nullptr;
        int                   list_max = 0;
        bool                  list_far = false;
        row_extra             ex{};
    };

    // The descriptor's 16-bit columns and column lists into a's fields.
    inline void use_c16(rv_args& a, const lal_csrmv_info* d)
    {
        a.c16      = d->d_c16;
        a.cbase    = d->d_cbase;
        a.lpos     = d->d_lpos;
        a.list     = d->d_list;
        a.lmeta    = d->d_lmeta;
        a.list_max = d->list_max;
        a.list_far = d->list_far;
    }

    int finish_partials(lal_context* c, int op, const post_args& a);
    template <typename T>
    int rowvec_launch(lal_context* c, int mode, const rv_args& a);
    // True where rowvec_launch has a kernel for this *_DOT mode and matrix.
    bool rowvec_can_dot(int mode, const rv_args& a);
}
