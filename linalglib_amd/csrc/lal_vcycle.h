// Internal launchers for the smoothers, coarse solves and PCG updates.
#pragma once

#include "lal_rowvec.h"

namespace lal
{
    // Device scalar slots of one solver (an array of LAL_SOLVER_SLOTS doubles).
    enum
    {
        S_GAMMA  = 0, // <z, r>, two generations
        S_ALPHA  = 2,
        S_RNORM  = 4, // inf-norm of the recursively updated residual
        S_RNORM0 = 5,
        S_TMP    = 6,
        LAL_SOLVER_SLOTS = 8
    };

    int csrmv_f64(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz, double alpha,
                  const int* rp, const int* ci, const double* v, const double* x, double beta,
                  double* y);
    int csrmv_f32(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz, float alpha,
                  const int* rp, const int* ci, const float* v, const float* x, float beta,
                  float* y);
    int residual_f64(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz,
                     const int* rp, const int* ci, const double* v, const double* x,
                     const double* b, double* r);
    int residual_f32(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz,
                     const int* rp, const int* ci, const float* v, const float* x,
                     const float* b, float* r);
    int csrmv_analysis_dev(lal_context* c, int m, int n, int nnz, const int* rp, const int* ci,
                           int exact, lal_csrmv_info** out);

    inline int csrmv(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz,
                     double alpha, const int* rp, const int* ci, const double* v,
                     const double* x, double beta, double* y)
    {
        return csrmv_f64(c, d, m, n, nnz, alpha, rp, ci, v, x, beta, y);
    }
    inline int csrmv(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz,
                     double alpha, const int* rp, const int* ci, const float* v, const float* x,
                     double beta, float* y)
    {
        return csrmv_f32(c, d, m, n, nnz, (float)alpha, rp, ci, v, x, (float)beta, y);
    }

    // Grid of the PCG reduction kernels, and of the update kernels at most
    // (one partial per block).
    constexpr int PCG_BLOCKS = 512;
    inline int update_blocks(int n)
    {
        return grid_for(n, SPMV_THREADS, PCG_BLOCKS);
    }

    template <typename T>
    int jacobi_sweep(lal_context* c, const lal_csrmv_info* d, int m, const int* rp,
                     const int* ci, const T* v, const T* diag, const T* dinv, const T* xold,
                     const T* b, T* xnew);
    // r = b - A x and y = x + r / a_ii: the residual a V-cycle restricts and
    // the Jacobi sweep that its post-smoothing builds on (fast descriptors).
    template <typename T>
    int residual_smoothed(lal_context* c, const lal_csrmv_info* d, int m, const int* rp,
                          const int* ci, const T* v, const T* x, const T* dinv, const T* b, T* r,
                          T* y, const post_args& post = {});
    // out = y + Q e (fast descriptors); with ex.part also <ex.w, out>'s partials
    // (can_add_dot)
    template <typename T>
    int add_product(lal_context* c, const lal_csrmv_info* d, int m, const int* rp, const int* ci,
                    const T* v, const T* e, const T* y, T* out, const row_extra& ex = {});
    template <typename T>
    bool can_add_dot(const lal_csrmv_info* d, int m, const int* rp, const int* ci, const T* v);
    // p' = z + beta p, y = A p' and *count partials of <y, p'>, beta = gamma_new /
    // gamma_old with gamma_new from its partials (as update_p, then product_dot);
    // *done false: not a matrix the one kernel takes, nothing was launched.
    template <typename T>
    int step_dot(lal_context* c, const lal_csrmv_info* d, int m, int n, const int* rp,
                 const int* ci, const T* v, const T* z, const T* p, T* p_new, T* y,
                 const double* part_g, int n_g, const double* gamma_old, double* gamma_new,
                 double* part, int* count, bool* done);
    // y = A x and *count partials of <y, x> in part (PCG_PARTS at most)
    template <typename T>
    int product_dot(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz, const int* rp,
                    const int* ci, const T* v, const T* x, T* y, double* part, int* count);
    // A level's arrays for make_ready: from A, d (the last diagonal entry of each
    // row), dinv = 1/d and, with v32, the FP32 copies of A's values, d and 1/d;
    // with qv, A P's values become those of Q = P - D^-1 A P (pattern of A P, a
    // superset of P's; both with ascending columns), in qv32 (or null) in FP32.
    struct ready_level
    {
        int           m;
        const int *   rp, *ci;
        const double* v;
        double *      d, *dinv;
        float *       v32, *d32, *dinv32;
        const int *   qrp, *qci;
        double*       qv;
        float*        qv32;
        const int *   prp, *pci;
        const double* pv;
    };
    // nnz: the longer of A's and Q's, which picks the lanes per row
    int make_ready(lal_context* c, const ready_level& a, long nnz);
    // y = (float) x for the arrays added.
    struct f32_copies
    {
        static constexpr int PER = 2048; // entries per workgroup
        struct one
        {
            const double* x;
            float*        y;
            size_t        len;
            int           block0;
        };
        one  c[40]; // (P and R of up to 20 levels)
        int  n = 0, blocks = 0;
        void add(const double* x, float* y, size_t len)
        {
            if(len == 0)
                return;
            c[n++] = {x, y, len, blocks};
            blocks += (int)((len + PER - 1) / PER);
        }
    };
    int copy_f32(lal_context* c, const f32_copies& a);
    template <typename T>
    int jacobi0_residual(lal_context* c, const lal_csrmv_info* d, int m, const int* rp,
                         const int* ci, const T* v, const T* diag, const T* dinv, const T* b,
                         T* x, T* r);
    template <typename T>
    int coarse_scalar(lal_context* c, const T* v, const T* b, T* x);
    template <typename T>
    int coarse_gs(lal_context* c, int n, const int* rp, const int* ci, const T* v, const T* b,
                  T* x);
    template <typename T>
    int coarse_dense(lal_context* c, int n, const double* inv, const T* b, T* x);
    // `sweeps` sequential Gauss-Seidel sweeps on x as given (one lane).
    int coarse_gs_sweeps(lal_context* c, int n, const int* rp, const int* ci, const double* v,
                         const double* b, double* x, int sweeps);
    // PCG_BLOCKS partials of <x, y> / max|x| (FP64 accumulation).
    template <typename TX, typename TY>
    int dot_partials(lal_context* c, int n, const TX* x, const TY* y, double* part);
    template <typename T>
    int norm_partials(lal_context* c, int n, const T* x, double* part);
    // op 0: sum, 1: max of a reduction's partials (post_args)
    int finish_partials(lal_context* c, int op, const post_args& a);
    // alpha = *gamma / sum of part_pq; x += alpha p, r -= alpha q,
    // update_blocks(n) partials of max|r|; with x0 also
    // x0 = (S)(r * rs_scale) * dinv, with rs also rs = (S)(r * rs_scale) (the
    // preconditioner's precision S; rs_scale = 1 leaves r as it is).
    template <typename T, typename S>
    int update_xr(lal_context* c, int n, const T* p, const T* q, T* x, T* r,
                  const double* part_pq, int n_pq, const double* gamma, double* part_r,
                  double* s_alpha, const S* dinv, S* x0, S* rs, double rs_scale = 1.0);
    // x = b * dinv
    template <typename T>
    int mul_elem(lal_context* c, int n, const T* b, const T* dinv, T* x);
    // b_c = R r and x_c = b_c * dinv_c (fast path only: needs a descriptor)
    template <typename T>
    int restrict_init(lal_context* c, const lal_csrmv_info* d, int m, const int* rp,
                      const int* ci, const T* v, const T* r, const T* dinv_c, T* b_c, T* x_c);
    // *gamma_new = sum of part_new; p = z + (*gamma_new / *gamma_old) p
    template <typename TZ, typename T>
    int update_p(lal_context* c, int n, const TZ* z, T* p, const double* part_new, int n_new,
                 const double* gamma_old, double* gamma_new);
    int scale_cast_f64_f32(lal_context* c, int n, const double* x, double scale, float* y);
    int axpy_f32_f64(lal_context* c, int n, double alpha, const float* d, double* x);
}
