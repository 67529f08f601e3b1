// V-cycle kernels: Jacobi smoothing (from zero, fused with the residual, and
// general sweeps), the coarse-level solves, and the PCG vector updates.
//
// Smoother arithmetic follows iterative_solvers/classic/jacobi.cpp:43-75:
// sigma = sigma + a_jk*xold_k over k != j in CSR order (two roundings per
// term), x_j = (b_j - sigma)/a_jj with a_jj the row's last diagonal entry.  A
// sweep from x = 0 gives sigma = +0 exactly, so it is x_j = b_j/a_jj; the
// fused kernel recomputes the neighbours' x_k = b_k/a_kk on the fly, which is
// bit-identical to smoothing first and forming r = b - A x afterwards.  These
// row-block kernels are the exact path; the fast path (lal_rowvec.hip) forms
// the same sweep as x + (b - A x) / a_ii.
//
// PCG reductions never use atomics or device-scope fences (on a multi-XCD
// part a device-scope release writes the L2 back, which costs more than the
// reduction itself).  Each reduction kernel writes one partial per block;
// the kernels that need the scalar re-reduce the partials themselves, every
// block in the same fixed order, so all blocks see bitwise the same value.
#include "lal_vcycle.h"

#include <type_traits>

namespace
{
    using lal::SPMV_THREADS;
    constexpr int RB = lal::PCG_BLOCKS;

    // MODE 0: x_new = Jacobi sweep of xold ; MODE 1: x = b/d and r = b - A x
    template <typename T, int MODE>
    __global__ void __launch_bounds__(SPMV_THREADS)
        jacobi_kernel(const int* __restrict__ blocks, int nb, int m, const int* __restrict__ rp,
                      const int* __restrict__ ci, const T* __restrict__ val,
                      const T* __restrict__ xold, const T* __restrict__ d,
                      const T* __restrict__ b, T* __restrict__ xnew, T* __restrict__ r,
                      int exact)
    {
        constexpr int CAP = lal::spmv_cap<T>::value;
        __shared__ T   s_v[CAP];
        __shared__ T   s_x[CAP];
        __shared__ int s_c[MODE == 0 ? CAP : 1];
        __shared__ int s_rp[SPMV_THREADS + 1];

        const int tid  = threadIdx.x;
        const int tile = lal::xcd_tile(blockIdx.x, nb);
        int       r0, r1;
        lal::block_rows(blocks, m, tile, &r0, &r1);
        const int nrows = r1 - r0;
        for(int i = tid; i <= nrows; i += SPMV_THREADS)
            s_rp[i] = rp[r0 + i];
        __syncthreads();

        const int  base   = s_rp[0];
        const int  end    = s_rp[nrows];
        const int  g      = lal::spmv_group(nrows, exact);
        const int  lrow   = tid / g;
        const int  lig    = tid & (g - 1);
        const bool active = lrow < nrows;
        const int  row    = r0 + lrow;
        const int  rs     = active ? s_rp[lrow] : 0;
        const int  re     = active ? s_rp[lrow + 1] : 0;

        T sigma = 0, ajj = 0;
        for(int cs = base; cs < end; cs += CAP)
        {
            const int len = min(CAP, end - cs);
#pragma unroll 4
            for(int k = tid; k < len; k += SPMV_THREADS)
            {
                const int c = ci[cs + k];
                s_v[k]      = val[cs + k];
                if(MODE == 0)
                {
                    s_c[k] = c;
                    s_x[k] = xold[c];
                }
                else
                    s_x[k] = b[c] / d[c];
            }
            __syncthreads();
            if(active)
            {
                const int a = max(rs, cs) - cs;
                const int e = min(re, cs + len) - cs;
                for(int j = a + lig; j < e; j += g)
                {
                    if(MODE == 0)
                    {
                        if(s_c[j] != row)
                            sigma = sigma + s_v[j] * s_x[j];
                        else
                            ajj = s_v[j];
                    }
                    else
                        sigma = sigma + s_v[j] * s_x[j];
                }
            }
            __syncthreads();
        }
        if(g > 1)
        {
            sigma = lal::group_sum(sigma, g);
            if(MODE == 0)
                ajj = lal::group_sum(ajj, g);
        }
        if(active && lig == 0)
        {
            if(MODE == 0)
                xnew[row] = (b[row] - sigma) / ajj;
            else
            {
                xnew[row] = b[row] / d[row];
                r[row]    = b[row] - sigma;
            }
        }
    }

    // Coarsest level with one unknown: x = b / a (amg.cpp:211-216).
    template <typename T>
    __global__ void scalar_solve_kernel(const T* __restrict__ val, const T* __restrict__ b,
                                        T* __restrict__ x)
    {
        if(threadIdx.x == 0 && blockIdx.x == 0)
            x[0] = b[0] / val[0];
    }

    // 1000 in-place Gauss-Seidel sweeps from x = 0 (amg.cpp:236-264), one lane.
    template <typename T>
    __global__ void __launch_bounds__(64)
        coarse_gs_kernel(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                         const T* __restrict__ val, const T* __restrict__ b, T* __restrict__ x,
                         int sweeps, int zero)
    {
        // The sweeps are one lane's sequential loop; when the operator, x and
        // b fit, the workgroup first stages them in LDS so that the loop's
        // dependent loads are LDS reads instead of L2 round trips.
        constexpr int          CGS_LDS = 40 * 1024;
        __shared__ __align__(16) unsigned char s_mem[CGS_LDS];
        const int              nnz  = rp[n];
        const size_t           need = sizeof(T) * ((size_t)nnz + 2 * (size_t)n)
                            + sizeof(int) * ((size_t)n + 1 + (size_t)nnz);
        const int tid = threadIdx.x;
        if(need <= CGS_LDS)
        {
            T*   s_v  = reinterpret_cast<T*>(s_mem);
            T*   s_x  = s_v + nnz;
            T*   s_b  = s_x + n;
            int* s_rp = reinterpret_cast<int*>(s_b + n);
            int* s_ci = s_rp + n + 1;
            for(int k = tid; k < nnz; k += blockDim.x)
            {
                s_v[k]  = val[k];
                s_ci[k] = ci[k];
            }
            for(int j = tid; j < n; j += blockDim.x)
            {
                s_x[j] = zero ? T(0) : x[j];
                s_b[j] = b[j];
            }
            for(int j = tid; j <= n; j += blockDim.x)
                s_rp[j] = rp[j];
            __syncthreads();
            if(tid == 0)
                for(int it = 0; it < sweeps; it++)
                    for(int j = 0; j < n; j++)
                    {
                        T sigma = 0, ajj = 0;
                        for(int k = s_rp[j]; k < s_rp[j + 1]; k++)
                        {
                            const int col = s_ci[k];
                            const T   v   = s_v[k];
                            if(col != j)
                                sigma = sigma + v * s_x[col];
                            else
                                ajj = v;
                        }
                        s_x[j] = (s_b[j] - sigma) / ajj;
                    }
            __syncthreads();
            for(int j = tid; j < n; j += blockDim.x)
                x[j] = s_x[j];
            return;
        }
        if(tid != 0)
            return;
        if(zero)
            for(int j = 0; j < n; j++)
                x[j] = 0;
        for(int it = 0; it < sweeps; it++)
            for(int j = 0; j < n; j++)
            {
                T sigma = 0, ajj = 0;
                for(int k = rp[j]; k < rp[j + 1]; k++)
                {
                    int col = ci[k];
                    T   v   = val[k];
                    if(col != j)
                        sigma = sigma + v * x[col];
                    else
                        ajj = v;
                }
                x[j] = (b[j] - sigma) / ajj;
            }
    }

    // Dense coarse solve x = Ainv b with the inverse kept in FP64.
    template <typename T>
    __global__ void __launch_bounds__(256)
        dense_apply_kernel(int n, const double* __restrict__ inv, const T* __restrict__ b,
                           T* __restrict__ x)
    {
        const int row  = blockIdx.x * 4 + (threadIdx.x >> 6);
        const int lane = threadIdx.x & 63;
        if(row >= n)
            return;
        double s = 0.0;
        for(int k = lane; k < n; k += 64)
            s = fma(inv[(size_t)row * n + k], (double)b[k], s);
        s = lal::wave_sum(s);
        if(lane == 0)
            x[row] = (T)s;
    }

    // ---------------------------------------------------- PCG vector updates
    using lal::block_total;
    using lal::combine;

    // part[block] = partial of sum x_i*y_i (OP 0) or max |x_i| (OP 1); x and y
    // may differ in precision (FP32 preconditioned vector, FP64 residual).
    template <typename TX, typename TY, int OP>
    __global__ void __launch_bounds__(SPMV_THREADS)
        partial_kernel(int n, const TX* __restrict__ x, const TY* __restrict__ y,
                       double* __restrict__ part)
    {
        double    acc    = 0.0;
        const int stride = gridDim.x * SPMV_THREADS;
        int       i      = blockIdx.x * SPMV_THREADS + threadIdx.x;
        for(; i + 3 * stride < n; i += 4 * stride)
        {
            TX a[4];
            TY b[4];
#pragma unroll
            for(int k = 0; k < 4; k++)
            {
                a[k] = x[i + k * stride];
                b[k] = OP == 0 ? y[i + k * stride] : (TY)a[k];
            }
#pragma unroll
            for(int k = 0; k < 4; k++)
                acc = OP == 0 ? acc + (double)a[k] * (double)b[k]
                              : combine<1>(acc, fabs((double)a[k]));
        }
        for(; i < n; i += stride)
            acc = OP == 0 ? acc + (double)x[i] * (double)y[i] : combine<1>(acc, fabs((double)x[i]));
        const double t = block_total<OP>(acc);
        if(threadIdx.x == 0)
            part[blockIdx.x] = t;
    }

    template <int OP>
    __global__ void __launch_bounds__(SPMV_THREADS) finish_kernel(lal::post_args a)
    {
        lal::post_block<OP>(a);
    }

    // alpha = gamma / <q, p>; x += alpha p; r += (-1*alpha) q (cg.cpp:185-193);
    // part_r[block] = max |r_i|.
    // When x0 is given, also x0 = r * dinv: the first Jacobi iterate from zero
    // of the preconditioner applied next to r, in the preconditioner's
    // precision S; when rs is given, rs = (S) r, the preconditioner's input.
    template <typename T, typename S>
    __global__ void __launch_bounds__(SPMV_THREADS)
        update_xr_kernel(int n, const T* __restrict__ p, const T* __restrict__ q,
                         T* __restrict__ x, T* __restrict__ r,
                         const double* __restrict__ part_pq, int n_pq,
                         const double* __restrict__ gamma, double* __restrict__ part_r,
                         double* __restrict__ s_alpha, const S* __restrict__ dinv,
                         S* __restrict__ x0, S* __restrict__ rs, T rs_scale)
    {
        const int stride = gridDim.x * SPMV_THREADS;
        int       i      = blockIdx.x * SPMV_THREADS + threadIdx.x;
        const double pq    = lal::total_of<0>(part_pq, n_pq);
        const double alpha = *gamma / pq;
        if(blockIdx.x == 0 && threadIdx.x == 0)
            *s_alpha = alpha;
        const T a  = (T)alpha;
        const T ma = (T)(-1.0 * alpha);
        double  acc = 0.0;
        auto    upd = [&](T pi, T qi, T xi, T ri, S di, int at) {
            x[at]    = a == (T)1 ? pi + xi : a * pi + xi;
            T rn     = ma == (T)1 ? qi + ri : ma * qi + ri;
            r[at]    = rn;
            const S r_s = (S)(rn * rs_scale);
            if(rs)
                rs[at] = r_s;
            if(x0)
                x0[at] = r_s * di;
            acc = combine<1>(acc, fabs((double)rn));
        };
        for(; i + 3 * stride < n; i += 4 * stride)
        {
            T pp[4], qq[4], xx[4], rr[4];
            S dd[4];
#pragma unroll
            for(int k = 0; k < 4; k++)
            {
                pp[k] = p[i + k * stride];
                qq[k] = q[i + k * stride];
                xx[k] = x[i + k * stride];
                rr[k] = r[i + k * stride];
                dd[k] = x0 ? dinv[i + k * stride] : (S)0;
            }
#pragma unroll
            for(int k = 0; k < 4; k++)
                upd(pp[k], qq[k], xx[k], rr[k], dd[k], i + k * stride);
        }
        for(; i < n; i += stride)
            upd(p[i], q[i], x[i], r[i], x0 ? dinv[i] : (S)0, i);
        const double t = block_total<1>(acc);
        if(threadIdx.x == 0)
            part_r[blockIdx.x] = t;
    }

    // beta = gamma_new / gamma_old; p = 1*z + beta*p (cg.cpp:205-211); z may be
    // the FP32 output of an FP32 preconditioner.
    template <typename TZ, typename T>
    __global__ void __launch_bounds__(SPMV_THREADS)
        update_p_kernel(int n, const TZ* __restrict__ z, T* __restrict__ p,
                        const double* __restrict__ part_new, int n_new,
                        const double* __restrict__ gamma_old, double* __restrict__ gamma_new)
    {
        const double g_new = lal::total_of<0>(part_new, n_new);
        const double g_old = *gamma_old;
        if(blockIdx.x == 0 && threadIdx.x == 0)
            *gamma_new = g_new;
        const T      beta  = (T)(g_new / g_old);
        const int    stride = gridDim.x * SPMV_THREADS;
        int          i      = blockIdx.x * SPMV_THREADS + threadIdx.x;
        for(; i + 3 * stride < n; i += 4 * stride)
        {
            T zz[4], pp[4];
#pragma unroll
            for(int k = 0; k < 4; k++)
            {
                zz[k] = (T)z[i + k * stride];
                pp[k] = p[i + k * stride];
            }
#pragma unroll
            for(int k = 0; k < 4; k++)
                p[i + k * stride] = beta == (T)0 ? zz[k] : zz[k] + beta * pp[k];
        }
        for(; i < n; i += stride)
            p[i] = beta == (T)0 ? (T)z[i] : (T)z[i] + beta * p[i];
    }

    // A level's operator made ready for the cycle, G lanes per row in one pass:
    // the row's last diagonal entry d and 1/d; with A P given, its entry (i, c)
    // becomes Q's, P(i, c) - 1/d (A P)(i, c); all of it in FP32 too where asked
    // for.  The row of P lies in the group's registers (up to G entries; a longer
    // one is searched in memory) and is compared by shuffles, so a row's loads
    // are two short chains.  Bound by memory and, on small levels, by the launch:
    // as six passes per level (two diagonals, Q, three FP32 copies) it took
    // 0.82 ms over a 121^3 diffusion hierarchy, as this one and one for all the
    // copies of P and R 0.52.
    template <int G>
    __global__ void __launch_bounds__(256) ready_kernel(lal::ready_level a)
    {
        const int i = blockIdx.x * (256 / G) + (int)(threadIdx.x / G);
        if(i >= a.m)
            return;
        const int t  = (int)(threadIdx.x & (G - 1));
        const int rs = a.rp[i], re = a.rp[i + 1];
        const int s = a.qv ? a.qrp[i] : 0, e = a.qv ? a.qrp[i + 1] : 0;
        const int    ps = a.qv ? a.prp[i] : 0, pn = a.qv ? a.prp[i + 1] - ps : 0;
        const int    pc = t < pn ? a.pci[ps + t] : -1;
        const double pw = t < pn ? a.pv[ps + t] : 0.0;
        int          last = -1;
        for(int j = rs + t; j < re; j += G)
        {
            if(a.ci[j] == i)
                last = j;
            if(a.v32)
                a.v32[j] = (float)a.v[j];
        }
        last            = lal::group_fold<G>(last, [](int x, int y) { return max(x, y); });
        const double d  = last >= 0 ? a.v[last] : 0.0;
        const double di = 1.0 / d;
        if(t == 0)
        {
            a.d[i]    = d;
            a.dinv[i] = di;
            if(a.v32)
            {
                a.d32[i]    = (float)d;
                a.dinv32[i] = 1.0f / (float)d;
            }
        }
        for(int j0 = s; j0 < e; j0 += G)
        {
            const int    j = j0 + t;
            const int    c = j < e ? a.qci[j] : -1;
            const double w = j < e ? a.qv[j] : 0.0;
            double       p = 0.0;
            if(pn <= G)
            {
                int hit = -1;
                for(int u = 0; u < pn; u++)
                    hit = __shfl(pc, u, G) == c ? u : hit;
                p = __shfl(pw, hit < 0 ? 0 : hit, G);
                p = hit < 0 ? 0.0 : p;
            }
            else
            {
                int lo = ps, hi = ps + pn; // first entry of P's row at or after c
                while(lo < hi)
                {
                    const int mid = (lo + hi) >> 1;
                    if(a.pci[mid] < c)
                        lo = mid + 1;
                    else
                        hi = mid;
                }
                p = lo < ps + pn && a.pci[lo] == c ? a.pv[lo] : 0.0;
            }
            if(j < e)
            {
                const double q = p - di * w;
                a.qv[j]        = q;
                if(a.qv32)
                    a.qv32[j] = (float)q;
            }
        }
    }

    // FP32 copies of several arrays, one after the other in the grid.
    __global__ void __launch_bounds__(256) copies_kernel(lal::f32_copies a)
    {
        int k = 0;
        while(k + 1 < a.n && a.c[k + 1].block0 <= (int)blockIdx.x)
            k++;
        const lal::f32_copies::one o = a.c[k];
        const size_t at = (size_t)(blockIdx.x - o.block0) * lal::f32_copies::PER + threadIdx.x;
#pragma unroll
        for(int u = 0; u < lal::f32_copies::PER / 256; u++)
            if(at + 256 * u < o.len)
                o.y[at + 256 * u] = (float)o.x[at + 256 * u];
    }

    // x = b * dinv (first Jacobi iterate from zero)
    template <typename T>
    __global__ void __launch_bounds__(256)
        mul_kernel(int n, const T* __restrict__ b, const T* __restrict__ dinv,
                   T* __restrict__ x)
    {
        for(int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
            x[i] = b[i] * dinv[i];
    }

    // y32 = (float)(scale * x64): the refinement residual, normalised
    __global__ void __launch_bounds__(256)
        scale_cast_kernel(int n, const double* __restrict__ x, double scale,
                          float* __restrict__ y)
    {
        for(int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
            y[i] = (float)(scale * x[i]);
    }

    // x64 += alpha * (double) d32
    __global__ void __launch_bounds__(256)
        axpy_f32_f64_kernel(int n, double alpha, const float* __restrict__ d,
                            double* __restrict__ x)
    {
        for(int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
            x[i] = alpha * (double)d[i] + x[i];
    }

    __global__ void __launch_bounds__(256)
        sddmm_kernel(int m, const int* __restrict__ rp, const int* __restrict__ ci, double scale,
                     const double* __restrict__ u, const double* __restrict__ v,
                     double* __restrict__ out)
    {
        int i = blockIdx.x * 256 + threadIdx.x;
        if(i >= m)
            return;
        const double su = scale * u[i];
        for(int j = rp[i]; j < rp[i + 1]; j++)
            out[j] = su * v[ci[j]];
    }
}

namespace lal
{
    template <typename T>
    int jacobi_sweep(lal_context* c, const lal_csrmv_info* d, int m, const int* rp,
                     const int* ci, const T* v, const T* diag, const T* dinv, const T* xold,
                     const T* b, T* xnew)
    {
        if(m == 0)
            return LAL_OK;
        if(d && !d->exact)
        {
            rv_args a{m, d->nnz, d->by_nnz, d->d_blocks, d->nblocks, rp, ci, v, xold, dinv, b, xnew, nullptr, 0.0,
                      0.0, d->win};
            lal::use_c16(a, d);
            a.keep = d->keep;
            return rowvec_launch<T>(c, RV_JACOBI, a);
        }
        int nb = spmv_grid(d, m);
        jacobi_kernel<T, 0><<<nb, SPMV_THREADS, 0, c->stream>>>(
            d ? d->d_blocks : nullptr, nb, m, rp, ci, v, xold, nullptr, b, xnew, nullptr,
            1); // no fast descriptor: one lane per row
        LAL_LAUNCHED();
        (void)diag;
        return LAL_OK;
    }

    template <typename T>
    int residual_smoothed(lal_context* c, const lal_csrmv_info* d, int m, const int* rp,
                          const int* ci, const T* v, const T* x, const T* dinv, const T* b, T* r,
                          T* y, const post_args& post)
    {
        if(m == 0)
            return LAL_OK;
        rv_args a{m, d->nnz, d->by_nnz, d->d_blocks, d->nblocks, rp, ci, v, x, dinv, b, r, y, 0.0,
                  0.0, d->win};
        lal::use_c16(a, d);
        a.keep    = d->keep;
        a.ex.post = post;
        return rowvec_launch<T>(c, RV_SMOOTHED, a);
    }

    template <typename T>
    static rv_args add_args(const lal_csrmv_info* d, int m, const int* rp, const int* ci,
                            const T* v, const T* e, const T* y, T* out)
    {
        rv_args a{m, d->nnz, d->by_nnz, d->d_blocks, d->nblocks, rp, ci, v, e, nullptr, y, out,
                  nullptr, 0.0, 0.0, d->win};
        lal::use_c16(a, d);
        a.keep = d->keep;
        return a;
    }

    template <typename T>
    bool can_add_dot(const lal_csrmv_info* d, int m, const int* rp, const int* ci, const T* v)
    {
        return rowvec_can_dot(RV_ADD_DOT, add_args<T>(d, m, rp, ci, v, nullptr, nullptr, nullptr));
    }

    template <typename T>
    int add_product(lal_context* c, const lal_csrmv_info* d, int m, const int* rp, const int* ci,
                    const T* v, const T* e, const T* y, T* out, const row_extra& ex)
    {
        if(m == 0)
            return LAL_OK;
        rv_args a = add_args<T>(d, m, rp, ci, v, e, y, out);
        a.ex      = ex;
        return rowvec_launch<T>(c, ex.part ? RV_ADD_DOT : RV_ADD, a);
    }

    template <typename T>
    int step_dot(lal_context* c, const lal_csrmv_info* d, int m, int n, const int* rp,
                 const int* ci, const T* v, const T* z, const T* p, T* p_new, T* y,
                 const double* part_g, int n_g, const double* gamma_old, double* gamma_new,
                 double* part, int* count, bool* done)
    {
        *done = false;
        if(!d || d->exact || m != n)
            return LAL_OK;
        rv_args a{m, d->nnz, d->by_nnz, d->d_blocks, d->nblocks, rp, ci, v, z, p, nullptr, y,
                  p_new, 1.0, 0.0, d->win};
        lal::use_c16(a, d);
        a.keep           = d->keep;
        a.ex.part        = part;
        a.ex.gamma_part  = part_g;
        a.ex.gamma_count = n_g;
        a.ex.gamma_old   = gamma_old;
        a.ex.gamma_new   = gamma_new;
        if(!rowvec_can_dot(RV_STEP_DOT, a))
            return LAL_OK;
        *done  = true;
        *count = d->nblocks;
        return rowvec_launch<T>(c, RV_STEP_DOT, a);
    }

    template <typename T>
    int product_dot(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz, const int* rp,
                    const int* ci, const T* v, const T* x, T* y, double* part, int* count)
    {
        if(d && !d->exact && m == n)
        {
            rv_args a{m, d->nnz, d->by_nnz, d->d_blocks, d->nblocks, rp, ci, v, x, nullptr,
                      nullptr, y, nullptr, 1.0, 0.0, d->win};
            lal::use_c16(a, d);
            a.keep    = d->keep;
            a.ex.part = part;
            a.ex.w    = x;
            if(rowvec_can_dot(RV_SPMV_DOT, a))
            {
                *count = d->nblocks;
                return rowvec_launch<T>(c, RV_SPMV_DOT, a);
            }
        }
        LAL_TRY(csrmv(c, d, m, n, nnz, 1.0, rp, ci, v, x, 0.0, y));
        *count = PCG_BLOCKS;
        return dot_partials<T, T>(c, m, y, x, part);
    }

    int make_ready(lal_context* c, const ready_level& a, long nnz)
    {
        if(a.m == 0)
            return LAL_OK;
        const auto go = [&](auto g) {
            constexpr int G = decltype(g)::value;
            ready_kernel<G><<<grid_for(a.m, 256 / G), 256, 0, c->stream>>>(a);
        };
        // about two steps of the group per row
        if(nnz <= 16L * a.m)
            go(std::integral_constant<int, 8>{});
        else if(nnz <= 48L * a.m)
            go(std::integral_constant<int, 16>{});
        else
            go(std::integral_constant<int, 64>{});
        LAL_LAUNCHED();
        return LAL_OK;
    }

    int copy_f32(lal_context* c, const f32_copies& a)
    {
        if(a.blocks == 0)
            return LAL_OK;
        copies_kernel<<<a.blocks, 256, 0, c->stream>>>(a);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    template <typename T>
    int jacobi0_residual(lal_context* c, const lal_csrmv_info* d, int m, const int* rp,
                         const int* ci, const T* v, const T* diag, const T* dinv, const T* b,
                         T* x, T* r)
    {
        if(m == 0)
            return LAL_OK;
        if(d && !d->exact)
        {
            rv_args a{m, d->nnz, d->by_nnz, d->d_blocks, d->nblocks, rp, ci, v, nullptr, dinv, b, x, r, 0.0, 0.0, d->win};
            lal::use_c16(a, d);
            a.keep = d->keep;
            return rowvec_launch<T>(c, RV_JACOBI0, a);
        }
        int nb = spmv_grid(d, m);
        jacobi_kernel<T, 1><<<nb, SPMV_THREADS, 0, c->stream>>>(
            d ? d->d_blocks : nullptr, nb, m, rp, ci, v, nullptr, diag, b, x, r,
            1); // no fast descriptor: one lane per row
        LAL_LAUNCHED();
        return LAL_OK;
    }

    template <typename T>
    int coarse_scalar(lal_context* c, const T* v, const T* b, T* x)
    {
        scalar_solve_kernel<T><<<1, 64, 0, c->stream>>>(v, b, x);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    template <typename T>
    int coarse_gs(lal_context* c, int n, const int* rp, const int* ci, const T* v, const T* b,
                  T* x)
    {
        coarse_gs_kernel<T><<<1, 64, 0, c->stream>>>(n, rp, ci, v, b, x, 1000, 1);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    int coarse_gs_sweeps(lal_context* c, int n, const int* rp, const int* ci, const double* v,
                         const double* b, double* x, int sweeps)
    {
        coarse_gs_kernel<double><<<1, 64, 0, c->stream>>>(n, rp, ci, v, b, x, sweeps, 0);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    template <typename T>
    int coarse_dense(lal_context* c, int n, const double* inv, const T* b, T* x)
    {
        dense_apply_kernel<T><<<(n + 3) / 4, 256, 0, c->stream>>>(n, inv, b, x);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    template <typename TX, typename TY>
    int dot_partials(lal_context* c, int n, const TX* x, const TY* y, double* part)
    {
        partial_kernel<TX, TY, 0><<<RB, SPMV_THREADS, 0, c->stream>>>(n, x, y, part);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    template <typename T>
    int norm_partials(lal_context* c, int n, const T* x, double* part)
    {
        partial_kernel<T, T, 1><<<RB, SPMV_THREADS, 0, c->stream>>>(n, x, x, part);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    int finish_partials(lal_context* c, int op, const post_args& a)
    {
        if(op == 0)
            finish_kernel<0><<<1, SPMV_THREADS, 0, c->stream>>>(a);
        else
            finish_kernel<1><<<1, SPMV_THREADS, 0, c->stream>>>(a);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    template <typename T, typename S>
    int update_xr(lal_context* c, int n, const T* p, const T* q, T* x, T* r,
                  const double* part_pq, int n_pq, const double* gamma, double* part_r,
                  double* s_alpha, const S* dinv, S* x0, S* rs, double rs_scale)
    {
        update_xr_kernel<T, S><<<update_blocks(n), SPMV_THREADS, 0, c->stream>>>(
            n, p, q, x, r, part_pq, n_pq, gamma, part_r, s_alpha, dinv, x0, rs, (T)rs_scale);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    template <typename T>
    int mul_elem(lal_context* c, int n, const T* b, const T* dinv, T* x)
    {
        if(n == 0)
            return LAL_OK;
        mul_kernel<T><<<grid_for(n, 256, 16384), 256, 0, c->stream>>>(n, b, dinv, x);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    template <typename T>
    int restrict_init(lal_context* c, const lal_csrmv_info* d, int m, const int* rp,
                      const int* ci, const T* v, const T* r, const T* dinv_c, T* b_c, T* x_c)
    {
        if(m == 0)
            return LAL_OK;
        rv_args a{m, d->nnz, d->by_nnz, d->d_blocks, d->nblocks, rp, ci, v, r, dinv_c, nullptr, b_c, x_c, 1.0, 0.0, d->win};
        lal::use_c16(a, d);
        a.keep = d->keep;
        return rowvec_launch<T>(c, RV_RESTRICT, a);
    }

    template <typename TZ, typename T>
    int update_p(lal_context* c, int n, const TZ* z, T* p, const double* part_new, int n_new,
                 const double* gamma_old, double* gamma_new)
    {
        update_p_kernel<TZ, T><<<update_blocks(n), SPMV_THREADS, 0, c->stream>>>(
            n, z, p, part_new, n_new, gamma_old, gamma_new);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    int scale_cast_f64_f32(lal_context* c, int n, const double* x, double scale, float* y)
    {
        scale_cast_kernel<<<grid_for(n, 256, 16384), 256, 0, c->stream>>>(n, x, scale, y);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    int axpy_f32_f64(lal_context* c, int n, double alpha, const float* d, double* x)
    {
        axpy_f32_f64_kernel<<<grid_for(n, 256, 16384), 256, 0, c->stream>>>(n, alpha, d, x);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    int sddmm(lal_context* c, int m, const int* rp, const int* ci, double scale, const double* u,
              const double* v, double* out)
    {
        if(m == 0)
            return LAL_OK;
        sddmm_kernel<<<grid_for(m, 256), 256, 0, c->stream>>>(m, rp, ci, scale, u, v, out);
        LAL_LAUNCHED();
        return LAL_OK;
    }

#define LAL_INST(T)                                                                          \
    template int jacobi_sweep<T>(lal_context*, const lal_csrmv_info*, int, const int*,       \
                                 const int*, const T*, const T*, const T*, const T*,         \
                                 const T*, T*);                                              \
    template int jacobi0_residual<T>(lal_context*, const lal_csrmv_info*, int, const int*,   \
                                     const int*, const T*, const T*, const T*, const T*, T*, \
                                     T*);                                                    \
    template int residual_smoothed<T>(lal_context*, const lal_csrmv_info*, int, const int*,  \
                                      const int*, const T*, const T*, const T*, const T*,    \
                                      T*, T*, const post_args&);                             \
    template int add_product<T>(lal_context*, const lal_csrmv_info*, int, const int*,        \
                                const int*, const T*, const T*, const T*, T*,                \
                                const row_extra&);                                           \
    template bool can_add_dot<T>(const lal_csrmv_info*, int, const int*, const int*,         \
                                 const T*);                                                  \
    template int step_dot<T>(lal_context*, const lal_csrmv_info*, int, int, const int*,     \
                             const int*, const T*, const T*, const T*, T*, T*,              \
                             const double*, int, const double*, double*, double*, int*,      \
                             bool*);                                                         \
    template int product_dot<T>(lal_context*, const lal_csrmv_info*, int, int, int,          \
                                const int*, const int*, const T*, const T*, T*, double*,     \
                                int*);                                                       \
    template int coarse_scalar<T>(lal_context*, const T*, const T*, T*);                     \
    template int coarse_gs<T>(lal_context*, int, const int*, const int*, const T*, const T*, \
                              T*);                                                           \
    template int coarse_dense<T>(lal_context*, int, const double*, const T*, T*);            \
    template int dot_partials<T, T>(lal_context*, int, const T*, const T*, double*);         \
    template int norm_partials<T>(lal_context*, int, const T*, double*);                     \
    template int update_xr<T, T>(lal_context*, int, const T*, const T*, T*, T*,              \
                                 const double*, int, const double*, double*, double*,        \
                                 const T*, T*, T*, double);                                  \
    template int update_p<T, T>(lal_context*, int, const T*, T*, const double*, int,         \
                                const double*, double*);                                     \
    template int mul_elem<T>(lal_context*, int, const T*, const T*, T*);                     \
    template int restrict_init<T>(lal_context*, const lal_csrmv_info*, int, const int*,      \
                                  const int*, const T*, const T*, const T*, T*, T*);
    LAL_INST(double)
    LAL_INST(float)
#undef LAL_INST
    // FP64 Krylov vectors with an FP32 preconditioner
    template int dot_partials<float, double>(lal_context*, int, const float*, const double*,
                                             double*);
    template int update_xr<double, float>(lal_context*, int, const double*, const double*,
                                          double*, double*, const double*, int,
                                          const double*, double*, double*, const float*, float*,
                                          float*, double);
    template int update_p<float, double>(lal_context*, int, const float*, double*,
                                         const double*, int, const double*, double*);
}

extern "C" int lal_sddmm_f64(lal_handle c, int m, int nnz, const int* rp, const int* ci,
                             double scale, const double* u, const double* v, double* vals)
{
    LAL_REQUIRE(c != nullptr && m >= 0 && nnz >= 0);
    LAL_REQUIRE(m == 0 || (rp && u && (nnz == 0 || (ci && v && vals))));
    return lal::sddmm(c, m, rp, ci, scale, u, v, vals);
}
