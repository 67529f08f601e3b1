// Fast CSR level kernels (see lal_rowvec.h).
#include "lal_rowvec.h"

namespace
{
    using lal::SPMV_THREADS;

    // The kernels' last argument: what its mode uses of a row_extra and no more.  A
    // launch copies its arguments to the device, and a small grid's V-cycle is its
    // launches: with 110 bytes more that nothing read, two pre-sweeps on 128^2
    // Poisson (31 launches) took 116 to 126 us in ten of eleven processes, without
    // them 94 to 96 in four of seven and 110 to 120 in the others; 20^2 Poisson 92 to
    // 102 and 71.
    struct no_extra
    {
    };
    template <int MODE>
    struct extra_for
    {
        using type = no_extra;
        static type of(const lal::row_extra&) { return {}; }
    };
    template <>
    struct extra_for<lal::RV_SMOOTHED>
    {
        using type = lal::post_args;
        static type of(const lal::row_extra& ex) { return ex.post; }
    };
    struct dot_extra
    {
        using type = lal::row_dot;
        static type of(const lal::row_extra& ex) { return ex; }
    };
    template <>
    struct extra_for<lal::RV_SPMV_DOT> : dot_extra
    {
    };
    template <>
    struct extra_for<lal::RV_ADD_DOT> : dot_extra
    {
    };
    template <>
    struct extra_for<lal::RV_STEP_DOT> : dot_extra
    {
    };
    template <int MODE>
    using mode_extra = typename extra_for<MODE>::type;

    // LDS bytes of a block's row starts (nrows + 1 <= SPMV_THREADS + 1 ints,
    // rounded up to 16 bytes so that the staged window stays aligned).
    constexpr int RP_LDS_BYTES = (int)(((SPMV_THREADS + 1) * sizeof(int) + 15) & ~15);

    template <typename T>
    __device__ __forceinline__ T stream_load(const T* p)
    {
        return __builtin_nontemporal_load(p);
    }

    typedef int            int4v __attribute__((ext_vector_type(4)));
    typedef unsigned short us4v __attribute__((ext_vector_type(4)));
    typedef float  flt4v __attribute__((ext_vector_type(4)));
    typedef double dbl2v __attribute__((ext_vector_type(2)));

    // Four consecutive matrix values read with 16-byte non-temporal loads.
    template <typename T>
    struct quad;
    template <>
    struct quad<float>
    {
        flt4v v;
        template <bool KEEP = false>
        __device__ __forceinline__ void load(const float* p)
        {
            if(KEEP)
                v = *reinterpret_cast<const flt4v*>(p);
            else
                v = __builtin_nontemporal_load(reinterpret_cast<const flt4v*>(p));
        }
        __device__ __forceinline__ void store(float* s) const
        {
            *reinterpret_cast<flt4v*>(s) = v;
        }
    };
    template <>
    struct quad<double>
    {
        dbl2v a, b;
        template <bool KEEP = false>
        __device__ __forceinline__ void load(const double* p)
        {
            if(KEEP)
            {
                a = reinterpret_cast<const dbl2v*>(p)[0];
                b = reinterpret_cast<const dbl2v*>(p)[1];
            }
            else
            {
                a = __builtin_nontemporal_load(reinterpret_cast<const dbl2v*>(p));
                b = __builtin_nontemporal_load(reinterpret_cast<const dbl2v*>(p) + 1);
            }
        }
        __device__ __forceinline__ void store(double* s) const
        {
            reinterpret_cast<dbl2v*>(s)[0] = a;
            reinterpret_cast<dbl2v*>(s)[1] = b;
        }
    };

    template <typename T, int MODE>
    __device__ __forceinline__ T gather(const T* __restrict__ x, const T* __restrict__ d,
                                        const T* __restrict__ b, int c, T beta = 0)
    {
        if(MODE == lal::RV_JACOBI0)
            return b[c] * d[c];
        if(MODE == lal::RV_STEP_DOT) // (as update_p_kernel)
            return beta == (T)0 ? x[c] : x[c] + beta * d[c];
        return x[c];
    }

    // What a row's epilogue reads besides its sum.  The staged kernels load it
    // with the block's first window, so that the row sums end in a store and
    // not in one more memory round trip.
    template <typename T>
    struct row_operands
    {
        T      b = 0, d = 0, x = 0, y = 0;
        double w = 0;
    };

    template <typename T, int MODE>
    __device__ __forceinline__ row_operands<T> load_operands(bool on, int row,
                                                             const T* __restrict__ x,
                                                             const T* __restrict__ d,
                                                             const T* __restrict__ b, T beta,
                                                             const T* __restrict__ y,
                                                             const mode_extra<MODE>& ex = {})
    {
        row_operands<T> o;
        if(!on)
            return o;
        if constexpr(MODE == lal::RV_SPMV_DOT || MODE == lal::RV_ADD_DOT)
            o.w = ex.wide ? static_cast<const double*>(ex.w)[row]
                          : (double)static_cast<const T*>(ex.w)[row];
        if(MODE == lal::RV_RESIDUAL || MODE == lal::RV_JACOBI || MODE == lal::RV_JACOBI0 ||
           MODE == lal::RV_SMOOTHED || MODE == lal::RV_ADD || MODE == lal::RV_ADD_DOT)
            o.b = b[row];
        if(MODE == lal::RV_JACOBI || MODE == lal::RV_JACOBI0 || MODE == lal::RV_RESTRICT ||
           MODE == lal::RV_SMOOTHED)
            o.d = d[row];
        if(MODE == lal::RV_JACOBI || MODE == lal::RV_SMOOTHED)
            o.x = x[row];
        if(MODE == lal::RV_SPMV && beta != (T)0)
            o.y = y[row];
        return o;
    }

    // y (and r) of one row from its sum acc = (A u)_row, per operation.
    template <typename T, int MODE>
    __device__ __forceinline__ void row_epilogue(int row, T acc, const row_operands<T>& o, T alpha,
                                                 T beta, T* __restrict__ y, T* __restrict__ r)
    {
        if(MODE == lal::RV_SPMV)
            y[row] = beta == (T)0 ? alpha * acc : fma(alpha, acc, beta * o.y);
        else if(MODE == lal::RV_RESTRICT)
        {
            y[row] = acc;
            r[row] = acc * o.d;
        }
        else if(MODE == lal::RV_RESIDUAL)
            y[row] = o.b - acc;
        else if(MODE == lal::RV_JACOBI)
            y[row] = o.x + (o.b - acc) * o.d;
        else if(MODE == lal::RV_SMOOTHED)
        {
            const T res = o.b - acc;
            y[row]      = res;
            r[row]      = o.x + res * o.d;
        }
        else if(MODE == lal::RV_ADD)
            y[row] = o.b + acc;
        else
        {
            y[row] = o.b * o.d;
            r[row] = o.b - acc;
        }
    }

    // The *_DOT epilogue, by the whole block: y of the lanes that end a row
    // (`head`), and the block's partial of <w, y> in FP64.
    template <typename T, int MODE>
    __device__ __forceinline__ void dot_epilogue(bool head, int row, T acc,
                                                 const row_operands<T>& o, T* __restrict__ y,
                                                 double* __restrict__ part)
    {
        const T v = MODE == lal::RV_ADD_DOT ? o.b + acc : acc;
        if(head)
            y[row] = v;
        const double t = lal::block_total<0>(head ? o.w * (double)v : 0.0);
        if(threadIdx.x == 0)
            *part = t;
    }

    template <typename T, int MODE>
    __global__ void __launch_bounds__(SPMV_THREADS)
        staged_kernel(int m, const int* __restrict__ blocks, int nb, const int* __restrict__ rp,
                      const int* __restrict__ ci, const T* __restrict__ val,
                      const T* __restrict__ x, const T* __restrict__ d,
                      const T* __restrict__ b, T alpha, T beta, T* __restrict__ y,
                      T* __restrict__ r)
    {
        constexpr int CAP = 2048;
        __shared__ T  s_p[CAP];

        const int tid  = threadIdx.x;
        const int tile = lal::xcd_tile(blockIdx.x, nb);
        int       r0, r1;
        lal::block_rows(blocks, m, tile, &r0, &r1);
        const int  nrows  = r1 - r0;
        const int  lg     = lal::spmv_group_log(nrows);
        const int  g      = 1 << lg;
        const int  lrow   = tid >> lg;
        const int  lig    = tid & (g - 1);
        const bool active = lrow < nrows;
        const int  row    = r0 + lrow;
        const int  base   = rp[r0];
        const int  end    = rp[r1];
        const int  rs     = active ? rp[row] : 0;
        const int  re     = active ? rp[row + 1] : 0;

        T acc = 0;
        for(int cs = base; cs < end; cs += CAP)
        {
            const int  len = min(CAP, end - cs);
            const int* cc  = ci + cs;
            const T*   vv  = val + cs;
            int        k   = tid;
            for(; k + 3 * SPMV_THREADS < len; k += 4 * SPMV_THREADS)
            {
                int c[4];
                T   v[4], xx[4];
#pragma unroll
                for(int u = 0; u < 4; u++)
                {
                    c[u] = stream_load(cc + k + u * SPMV_THREADS);
                    v[u] = stream_load(vv + k + u * SPMV_THREADS);
                }
#pragma unroll
                for(int u = 0; u < 4; u++)
                    xx[u] = gather<T, MODE>(x, d, b, c[u]);
#pragma unroll
                for(int u = 0; u < 4; u++)
                    s_p[k + u * SPMV_THREADS] = v[u] * xx[u];
            }
            for(; k < len; k += SPMV_THREADS)
                s_p[k] = stream_load(vv + k) * gather<T, MODE>(x, d, b, stream_load(cc + k));
            __syncthreads();
            if(active)
            {
                const int a = max(rs, cs) - cs;
                const int e = min(re, cs + len) - cs;
                for(int j = a + lig; j < e; j += g)
                    acc += s_p[j];
            }
            __syncthreads();
        }
        if(g > 1)
            acc = lal::group_sum(acc, g);
        if(!active || lig != 0)
            return;
        row_epilogue<T, MODE>(row, acc, load_operands<T, MODE>(true, row, x, d, b, beta, y), alpha,
                              beta, y, r);
    }

    // Row sum over the staged nonzeros [j, e) (stride g): UR column indices
    // and values come from LDS, then UR gathers are in flight at once.
    template <typename T, int MODE, int UR>
    __device__ __forceinline__ T staged_row_sum(const int* s_c, const T* s_v, int j, int e, int g,
                                                const T* __restrict__ x,
                                                const T* __restrict__ d,
                                                const T* __restrict__ b, T beta)
    {
        T acc = 0;
        if(j >= e)
            return acc;
        const int csafe = s_c[j];
        for(; j < e; j += UR * g)
        {
            int  cc[UR];
            T    vv[UR], xx[UR];
            bool ok[UR];
#pragma unroll
            for(int u = 0; u < UR; u++)
            {
                ok[u] = j + u * g < e;
                cc[u] = ok[u] ? s_c[j + u * g] : csafe;
                vv[u] = ok[u] ? s_v[j + u * g] : (T)0;
            }
#pragma unroll
            for(int u = 0; u < UR; u++)
                xx[u] = gather<T, MODE>(x, d, b, cc[u], beta);
#pragma unroll
            for(int u = 0; u < UR; u++)
            {
                const T p = vv[u] * xx[u];
                acc += ok[u] ? p : (T)0;
            }
        }
        return acc;
    }

    // Four consecutive column indices at q (a multiple of 4): 16 bytes of
    // int32, or 8 bytes of 16-bit offsets from the block's base cb.
    template <bool KEEP, bool C16>
    __device__ __forceinline__ int4v load_cols(const int* __restrict__ ci,
                                               const unsigned short* __restrict__ c16, int cb,
                                               int q)
    {
        if(C16)
        {
            const us4v* p = reinterpret_cast<const us4v*>(c16 + q);
            const us4v  w = KEEP ? *p : __builtin_nontemporal_load(p);
            return int4v{cb + (int)w.x, cb + (int)w.y, cb + (int)w.z, cb + (int)w.w};
        }
        const int4v* p = reinterpret_cast<const int4v*>(ci + q);
        return KEEP ? *p : __builtin_nontemporal_load(p);
    }

    // Quad-staged row-gather kernel (16-byte aligned ci and val).
    //
    // Phase 1 copies the block's column indices and values into LDS with
    // 16-byte non-temporal loads, four consecutive nonzeros per lane, over a
    // window aligned down to a multiple of four (WIN, a multiple of four, is
    // the widest such window of the matrix's blocks and at most CAP + 4
    // entries, so a block of at most CAP nonzeros always fits one window).  Phase 2 lets each
    // row (one lane, or G lanes for short blocks) walk its own nonzeros in LDS
    // and gather x itself: one gather instruction then covers the same
    // stencil offset of 64 consecutive rows, a few cache lines, instead of
    // every offset of a handful of rows.  Fewer and wider memory instructions
    // and compact gathers are what lift this kernel over the product-staging
    // one on CDNA.
    template <typename T, int MODE, bool KEEP, bool C16>
    __global__ void __launch_bounds__(SPMV_THREADS)
        quad_kernel(int m, int nnz, const int* __restrict__ blocks, int nb, int win,
                    const int* __restrict__ rp, const int* __restrict__ ci,
                    const unsigned short* __restrict__ c16, const int* __restrict__ cbase,
                    const T* __restrict__ val, const T* __restrict__ x,
                    const T* __restrict__ d, const T* __restrict__ b, T alpha, T beta,
                    T* __restrict__ y, T* __restrict__ r, mode_extra<MODE> ex)
    {
        if constexpr(MODE == lal::RV_SMOOTHED)
            if((int)blockIdx.x == nb)
            {
                // (the grid has this workgroup only with a reduction to finish)
                lal::post_block<1>(ex);
                return;
            }
        if constexpr(MODE == lal::RV_STEP_DOT)
        {
            const double g_new = lal::total_of<0>(ex.gamma_part, ex.gamma_count);
            if(blockIdx.x == 0 && threadIdx.x == 0)
                *ex.gamma_new = g_new;
            beta = (T)(g_new / *ex.gamma_old);
        }
        // the block's row starts, then win entries of columns, then win
        // values (win: a multiple of 4)
        extern __shared__ __attribute__((aligned(16))) unsigned char s_raw[];
        int* s_rp = reinterpret_cast<int*>(s_raw);
        int* s_c  = reinterpret_cast<int*>(s_raw + RP_LDS_BYTES);
        T*   s_v  = reinterpret_cast<T*>(s_raw + RP_LDS_BYTES + sizeof(int) * win);
        const int WIN = win;

        const int   tid  = threadIdx.x;
        const int   tile = lal::xcd_tile(blockIdx.x, nb);
        const int4v mt   = reinterpret_cast<const int4v*>(blocks + lal::block_meta_offset(nb))[tile];
        const int   r0 = mt.x, r1 = mt.y;
        const int  nrows  = r1 - r0;
        const int  lg     = lal::spmv_group_log(nrows);
        const int  g      = 1 << lg;
        const int  lrow   = tid >> lg;
        const int  lig    = tid & (g - 1);
        const bool active = lrow < nrows;
        const int  row    = r0 + lrow;
        const int  base   = mt.z;
        const int  end    = mt.w;
        const int  nnz4   = nnz & ~3;
        const int  cb     = C16 ? cbase[tile] : 0; // this block's 16-bit column base
        // The row bounds travel with the first window's loads (through LDS)
        // instead of being awaited before them: rp[r0] and rp[r1] are the
        // descriptor's base and end, lane i loads rp[r0 + i] for 0 < i < nrows.
        const int rpv = (tid > 0 && tid < nrows) ? rp[r0 + tid] : 0;
        const row_operands<T> ops =
            load_operands<T, MODE>(active && lig == 0, row, x, d, b, beta, y, ex);
        int       rs = 0, re = 0;
        bool      bounds = false;

        T acc = 0;
        for(int ws = base & ~3; ws < end; ws += WIN)
        {
            const int we   = min(ws + WIN, end);
            const int vend = min((we + 3) & ~3, nnz4); // quads inside the arrays
            for(int q0 = ws + 4 * tid; q0 < vend; q0 += 8 * SPMV_THREADS)
            {
                int4v   cq[2];
                quad<T> vq[2];
                int     qq[2];
#pragma unroll
                for(int u = 0; u < 2; u++)
                {
                    qq[u] = min(q0 + 4 * SPMV_THREADS * u, vend - 4);
                    cq[u] = load_cols<KEEP, C16>(ci, c16, cb, qq[u]);
                    vq[u].template load<KEEP>(val + qq[u]);
                }
                // Every quad is stored unconditionally: a lane whose second
                // quad lies past the window's end stores the window's last
                // quad again, the same values its owner stores.  A stored
                // value used only under a condition lets the compiler sink
                // its load into that branch, after the first quad's wait,
                // which makes two HBM round trips of one.
#pragma unroll
                for(int u = 0; u < 2; u++)
                {
                    *reinterpret_cast<int4v*>(s_c + (qq[u] - ws)) = cq[u];
                    vq[u].store(s_v + (qq[u] - ws));
                }
            }
            // the arrays' last nnz % 4 entries
            for(int k = max(vend, ws) + tid; k < we; k += SPMV_THREADS)
            {
                s_c[k - ws] = C16 ? cb + (int)c16[k] : ci[k];
                s_v[k - ws] = val[k];
            }
            if(!bounds)
            {
                if(tid > 0 && tid < nrows)
                    s_rp[tid] = rpv;
                if(tid == 0)
                {
                    s_rp[0]     = base;
                    s_rp[nrows] = end;
                }
            }
            __syncthreads();
            if(!bounds)
            {
                rs     = active ? s_rp[lrow] : 0;
                re     = active ? s_rp[lrow + 1] : 0;
                bounds = true;
            }
            if(active)
            {
                const int a = max(rs, ws) - ws + lig;
                const int e = min(re, we) - ws;
                acc += g == 1 ? staged_row_sum<T, MODE, 8>(s_c, s_v, a, e, 1, x, d, b, beta)
                              : staged_row_sum<T, MODE, 4>(s_c, s_v, a, e, g, x, d, b, beta);
            }
            __syncthreads();
        }
        if(g > 1)
            acc = lal::group_sum(acc, g);
        if constexpr(MODE == lal::RV_STEP_DOT)
        {
            const bool head = active && lig == 0;
            row_operands<T> o;
            if(head)
            {
                const T p = gather<T, MODE>(x, d, b, row, beta);
                r[row]    = p;
                o.w       = (double)p;
            }
            dot_epilogue<T, MODE>(head, row, acc, o, y, ex.part + tile);
            return;
        }
        if constexpr(MODE == lal::RV_SPMV_DOT)
        {
            dot_epilogue<T, MODE>(active && lig == 0, row, acc, ops, y, ex.part + tile);
            return;
        }
        if(!active || lig != 0)
            return;
        row_epilogue<T, MODE>(row, acc, ops, alpha, beta, y, r);
    }

    // Quad-staged kernel that gathers by nonzero (16-byte aligned ci and val):
    // each lane gathers x for the four consecutive nonzeros it loaded and
    // stores the products in LDS; the rows then sum their products.  Used for
    // the rectangular transfer operators, whose short and uneven rows would
    // leave lanes of the per-row gather idle.
    template <typename T, int MODE, bool C16>
    __global__ void __launch_bounds__(SPMV_THREADS)
        quad_nnz_kernel(int m, int nnz, const int* __restrict__ blocks, int nb, int win,
                        const int* __restrict__ rp, const int* __restrict__ ci,
                        const unsigned short* __restrict__ c16, const int* __restrict__ cbase,
                        const T* __restrict__ val, const T* __restrict__ x,
                        const T* __restrict__ d, const T* __restrict__ b, T alpha, T beta,
                        T* __restrict__ y, T* __restrict__ r)
    {
        // the block's row starts, then win products
        extern __shared__ __attribute__((aligned(16))) unsigned char s_raw[];
        int*      s_rp = reinterpret_cast<int*>(s_raw);
        T*        s_p  = reinterpret_cast<T*>(s_raw + RP_LDS_BYTES);
        const int WIN  = win;

        const int   tid  = threadIdx.x;
        const int   tile = lal::xcd_tile(blockIdx.x, nb);
        const int4v mt   = reinterpret_cast<const int4v*>(blocks + lal::block_meta_offset(nb))[tile];
        const int   r0 = mt.x, r1 = mt.y;
        const int  nrows  = r1 - r0;
        const int  lg     = lal::spmv_group_log(nrows);
        const int  g      = 1 << lg;
        const int  lrow   = tid >> lg;
        const int  lig    = tid & (g - 1);
        const bool active = lrow < nrows;
        const int  row    = r0 + lrow;
        const int  base   = mt.z;
        const int  end    = mt.w;
        const int  nnz4   = nnz & ~3;
        const int  cb     = C16 ? cbase[tile] : 0; // this block's 16-bit column base
        // row bounds through LDS, loaded with the first window (quad_kernel)
        const int rpv = (tid > 0 && tid < nrows) ? rp[r0 + tid] : 0;
        const row_operands<T> ops =
            load_operands<T, MODE>(active && lig == 0, row, x, d, b, beta, y);
        int       rs = 0, re = 0;
        bool      bounds = false;

        T acc = 0;
        for(int ws = base & ~3; ws < end; ws += WIN)
        {
            const int we   = min(ws + WIN, end);
            const int vend = min((we + 3) & ~3, nnz4);
            for(int q0 = ws + 4 * tid; q0 < vend; q0 += 8 * SPMV_THREADS)
            {
                // two quads per lane, both loaded before either's gathers (a
                // second quad past the window's end repeats its last quad and
                // stores the same products as that quad's owner)
                int4v   cq[2];
                quad<T> vq[2];
                int     qq[2];
#pragma unroll
                for(int u = 0; u < 2; u++)
                {
                    qq[u] = min(q0 + 4 * SPMV_THREADS * u, vend - 4);
                    cq[u] = load_cols<false, C16>(ci, c16, cb, qq[u]);
                    vq[u].load(val + qq[u]);
                    // a 16-bit column of a neighbouring block's entry (a quad
                    // straddling the block's ends) decodes against this
                    // block's base: gather at the base instead (its product
                    // belongs to no row of this block)
                    if(C16)
#pragma unroll
                        for(int e = 0; e < 4; e++)
                            if(qq[u] + e < base || qq[u] + e >= end)
                                cq[u][e] = cb;
                }
                T v8[8], x8[8];
#pragma unroll
                for(int u = 0; u < 2; u++)
                    vq[u].store(v8 + 4 * u);
#pragma unroll
                for(int u = 0; u < 2; u++)
#pragma unroll
                    for(int e = 0; e < 4; e++)
                        x8[4 * u + e] = gather<T, MODE>(x, d, b, cq[u][e]);
#pragma unroll
                for(int u = 0; u < 2; u++)
#pragma unroll
                    for(int e = 0; e < 4; e++)
                        s_p[qq[u] - ws + e] = v8[4 * u + e] * x8[4 * u + e];
            }
            for(int k = max(vend, ws) + tid; k < we; k += SPMV_THREADS)
                s_p[k - ws] = val[k] * gather<T, MODE>(x, d, b,
                                                       C16 ? (k < base ? cb : cb + (int)c16[k])
                                                           : ci[k]);
            if(!bounds)
            {
                if(tid > 0 && tid < nrows)
                    s_rp[tid] = rpv;
                if(tid == 0)
                {
                    s_rp[0]     = base;
                    s_rp[nrows] = end;
                }
            }
            __syncthreads();
            if(!bounds)
            {
                rs     = active ? s_rp[lrow] : 0;
                re     = active ? s_rp[lrow + 1] : 0;
                bounds = true;
            }
            if(active)
            {
                const int a = max(rs, ws) - ws + lig;
                const int e = min(re, we) - ws;
                for(int j = a; j < e; j += g)
                    acc += s_p[j];
            }
            __syncthreads();
        }
        if(g > 1)
            acc = lal::group_sum(acc, g);
        if(!active || lig != 0)
            return;
        row_epilogue<T, MODE>(row, acc, ops, alpha, beta, y, r);
    }

    // Sum of the staged products s_p[j], s_p[j + g], ... below e, four reads
    // in flight.
    template <typename T>
    __device__ __forceinline__ T product_sum(const T* s_p, int j, int e, int g)
    {
        T acc = 0;
        if(g == 1) // (uniform) constant offsets
        {
            for(; j + 3 < e; j += 4)
            {
                const T p0 = s_p[j], p1 = s_p[j + 1], p2 = s_p[j + 2], p3 = s_p[j + 3];
                acc += p0;
                acc += p1;
                acc += p2;
                acc += p3;
            }
            for(; j < e; j++)
                acc += s_p[j];
            return acc;
        }
        for(; j + 3 * g < e; j += 4 * g)
        {
            const T p0 = s_p[j], p1 = s_p[j + g], p2 = s_p[j + 2 * g], p3 = s_p[j + 3 * g];
            acc += p0;
            acc += p1;
            acc += p2;
            acc += p3;
        }
        for(; j < e; j += g)
            acc += s_p[j];
        return acc;
    }

    // p[i] with a 32-bit byte offset from a uniform base
    template <typename V, typename T>
    __device__ __forceinline__ V load_at(const T* p, unsigned byte)
    {
        return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(p) + byte);
    }
    template <typename V, bool KEEP, typename T>
    __device__ __forceinline__ V stream_at(const T* p, unsigned byte)
    {
        if(KEEP)
            return load_at<V>(p, byte);
        return __builtin_nontemporal_load(
            reinterpret_cast<const V*>(reinterpret_cast<const char*>(p) + byte));
    }

    // Row sums with x gathered through LDS, for operators whose blocks name
    // each column several times (a hierarchy's long-row operators).
    //
    // A gather of 64 scattered entries keeps the L1 busy for 34-38 clocks, one
    // of consecutive lanes' neighbouring entries for 5 (FP32) or 16 (FP64).  So
    // the block gathers its distinct columns once, in ascending order, into
    // LDS, while its values and the nonzeros' places in that list are on their
    // way; the lanes then form the products of the quads they loaded out of
    // LDS, and the rows sum theirs.  The instructions are what is left to pay
    // (30 vector instructions per nonzero of a lane kept the SIMDs busy for
    // half of the time): addresses are 32-bit offsets from the block's
    // uniform bases, places are stored as byte offsets, lane groups are
    // shifts.  Blocks hold at most 2044 nonzeros, 512 quads, so one window of two
    // quads per lane always does.
    // The lists are read two entries per lane: loads of 16 bits per lane cost as
    // much as scattered ones (128^3 level 1 in FP32: 31 us with them, 26 with
    // pairs).
    constexpr int LIST_U = 4; // list pairs per lane: a list has at most 2044 entries

    //
    // KEEP: the matrix is read with cache-allocating loads (lal_csrmv_info::keep).
    // FAR: some block's columns span more than 65536 (the finest restriction
    // of a large grid), and its list's entries from `split` on are 65536 further.
    template <typename T, int MODE, bool FAR, bool KEEP>
    __global__ void __launch_bounds__(SPMV_THREADS)
        list_kernel(const int* __restrict__ blocks, int nb, int list_max,
                    const int* __restrict__ rp, const unsigned short* __restrict__ lpos,
                    const unsigned short* __restrict__ list, const int* __restrict__ lmeta,
                    const T* __restrict__ val, const T* __restrict__ x, const T* __restrict__ d,
                    const T* __restrict__ b, T alpha, T beta, T* __restrict__ y,
                    T* __restrict__ r, mode_extra<MODE> ex)
    {
        typedef int int2v __attribute__((ext_vector_type(2)));
        // the block's row starts, its x entries, then its products
        extern __shared__ __attribute__((aligned(16))) unsigned char s_raw[];
        int* s_rp = reinterpret_cast<int*>(s_raw);
        T*   s_x  = reinterpret_cast<T*>(s_raw + RP_LDS_BYTES);
        T*   s_p  = s_x + list_max; // list_max: a multiple of 4

        const unsigned tid  = threadIdx.x;
        const int      tile = lal::xcd_tile(blockIdx.x, nb);
        const int4v mt = reinterpret_cast<const int4v*>(blocks + lal::block_meta_offset(nb))[tile];
        const int2v lm = reinterpret_cast<const int2v*>(lmeta)[tile];
        const int   r0 = mt.x, nrows = mt.y - mt.x, base = mt.z, end = mt.w;
        const unsigned len   = (unsigned)lm.x & 0xfffu;
        const unsigned split = (unsigned)lm.x >> 12 & 0xfffu; // entries from here on: 65536 further
        const int      lg    = lm.x >> 24;                    // log2 of the lanes per row
        const int      ws  = base & ~3;
        const unsigned nq  = (unsigned)(end - ws + 3) >> 2;
        // (JACOBI0's x is b d, as in gather())
        constexpr bool        ZERO = MODE == lal::RV_JACOBI0;
        const T*              xb = (ZERO ? b : x) + lm.y;
        const T*              db = ZERO ? d + lm.y : nullptr;
        const T*              vb = val + ws;
        const unsigned short* pb = lpos + ws;
        const unsigned short* lb = list + lal::list_start(base, tile);
        const unsigned        np = (len + 1) >> 1; // list pairs

        unsigned lo[LIST_U];
#pragma unroll
        for(int u = 0; u < LIST_U; u++)
            if(SPMV_THREADS * u < np) // (uniform)
                lo[u] = stream_at<unsigned, KEEP>(lb, 4u * min(tid + SPMV_THREADS * u, np - 1));
        us4v    pq[2];
        quad<T> vq[2];
#pragma unroll
        for(int u = 0; u < 2; u++)
            if(SPMV_THREADS * u < nq) // (uniform)
            {
                const unsigned q = min(tid + SPMV_THREADS * u, nq - 1);
                pq[u]            = stream_at<us4v, KEEP>(pb, 8u * q);
                vq[u].template load<KEEP>(reinterpret_cast<const T*>(
                    reinterpret_cast<const char*>(vb) + 4u * sizeof(T) * q));
            }
        const int  lrow = (int)tid >> lg;
        const bool on   = lrow < nrows;
        const bool head = on && (tid & ((1u << lg) - 1u)) == 0;
        const int  rpv  = rp[r0 + min((int)tid, nrows)];
        const row_operands<T> ops = load_operands<T, MODE>(head, r0 + lrow, x, d, b, beta, y, ex);
        const auto x_at = [&](unsigned at) {
            const unsigned byte = (unsigned)sizeof(T) * at;
            return ZERO ? load_at<T>(xb, byte) * load_at<T>(db, byte) : load_at<T>(xb, byte);
        };
        // (a list of odd length repeats its last column once more)
        T xv[LIST_U][2];
#pragma unroll
        for(int u = 0; u < LIST_U; u++)
            if(SPMV_THREADS * u < np)
            {
                unsigned o0 = lo[u] & 0xffffu, o1 = lo[u] >> 16;
                if(FAR)
                {
                    const unsigned i = 2u * min(tid + SPMV_THREADS * u, np - 1);
                    o0               = lal::list_offset(o0, i, split);
                    o1               = lal::list_offset(o1, i + 1, split);
                }
                xv[u][0] = x_at(o0);
                xv[u][1] = x_at(o1);
            }
#pragma unroll
        for(int u = 0; u < LIST_U; u++)
            if(SPMV_THREADS * u < np)
            {
                T* at = s_x + 2u * min(tid + SPMV_THREADS * u, np - 1);
                at[0] = xv[u][0];
                at[1] = xv[u][1];
            }
        if((int)tid < nrows)
            s_rp[tid] = rpv;
        if(tid == 0)
            s_rp[nrows] = end;
        __syncthreads();
        // (places of a neighbouring block's entries in the window's first and
        // last quad are below list_max too; their products belong to no row
        // here)
#pragma unroll
        for(int u = 0; u < 2; u++)
            if(SPMV_THREADS * u < nq)
            {
                T v[4], p[4];
                vq[u].store(v);
#pragma unroll
                for(int e = 0; e < 4; e++)
                    p[e] = v[e] * load_at<T>(s_x, (unsigned)(sizeof(T) / 4) * pq[u][e]);
                quad<T> out;
                out.template load<true>(p);
                out.store(s_p + 4u * min(tid + SPMV_THREADS * u, nq - 1));
            }
        __syncthreads();
        T acc = 0;
        if(on)
            acc = product_sum(s_p, s_rp[lrow] - ws + (int)(tid & ((1u << lg) - 1u)),
                              s_rp[lrow + 1] - ws, 1 << lg);
        if(lg > 0)
            acc = lal::group_sum(acc, 1 << lg);
        if constexpr(MODE == lal::RV_ADD_DOT)
            dot_epilogue<T, MODE>(head, r0 + lrow, acc, ops, y, ex.part + tile);
        else if(head)
            row_epilogue<T, MODE>(r0 + lrow, acc, ops, alpha, beta, y, r);
    }

    template <typename T>
    bool kept(const lal::rv_args& a)
    {
        return a.keep & (sizeof(T) == sizeof(double) ? 1 : 2);
    }

    template <typename T, int MODE, bool C16>
    void launch_quad(lal_context* c, const lal::rv_args& a, int nb)
    {
        // LDS sized to the widest block window of this matrix, so that short
        // blocks leave room for more resident workgroups
        const int    win  = a.win;
        auto*        fn   = kept<T>(a) ? quad_kernel<T, MODE, true, C16> : quad_kernel<T, MODE, false, C16>;
        const int    more = MODE == lal::RV_SMOOTHED && a.ex.post.part ? 1 : 0;
        fn<<<nb + more, SPMV_THREADS, RP_LDS_BYTES + (sizeof(int) + sizeof(T)) * win, c->stream>>>(
            a.m, a.nnz, a.blocks, nb, win, a.rp, a.ci, a.c16, a.cbase, (const T*)a.val,
            (const T*)a.x, (const T*)a.d, (const T*)a.b, (T)a.alpha, (T)a.beta, (T*)a.y, (T*)a.r,
            extra_for<MODE>::of(a.ex));
    }

    template <typename T, int MODE>
    void launch_list(lal_context* c, const lal::rv_args& a, int nb)
    {
        const int    lm  = (a.list_max + 3) & ~3;
        const size_t lds = RP_LDS_BYTES + sizeof(T) * (size_t)(lm + a.win);
        auto* fn = kept<T>(a) ? (a.list_far ? list_kernel<T, MODE, true, true>
                                        : list_kernel<T, MODE, false, true>)
                          : (a.list_far ? list_kernel<T, MODE, true, false>
                                        : list_kernel<T, MODE, false, false>);
        fn<<<nb, SPMV_THREADS, lds, c->stream>>>(
            a.blocks, nb, lm, a.rp, a.lpos, a.list, a.lmeta, (const T*)a.val, (const T*)a.x,
            (const T*)a.d, (const T*)a.b, (T)a.alpha, (T)a.beta, (T*)a.y, (T*)a.r,
            extra_for<MODE>::of(a.ex));
    }

    // Which kernel reads a matrix.
    enum
    {
        BY_STAGED, // unaligned arrays
        BY_LIST,   // x through LDS by column lists
        BY_NNZ,    // gathers over consecutive nonzeros
        BY_QUAD
    };
    int route(const lal::rv_args& a)
    {
        const bool val16 = (reinterpret_cast<uintptr_t>(a.val) & 15) == 0;
        const bool cols  = (a.c16 && a.cbase) || (reinterpret_cast<uintptr_t>(a.ci) & 15) == 0;
        if(!a.blocks || !val16)
            return BY_STAGED;
        if(a.list_max > 0)
            return BY_LIST;
        return !cols ? BY_STAGED : a.by_nnz ? BY_NNZ : BY_QUAD;
    }

    template <typename T, int MODE>
    int launch(lal_context* c, const lal::rv_args& a)
    {
        const int  nb  = a.blocks ? a.nb : (a.m + SPMV_THREADS - 1) / SPMV_THREADS;
        const int  by  = route(a);
        const bool c16 = a.c16 && a.cbase;
        if(a.ex.post.part && (MODE != lal::RV_SMOOTHED || by != BY_QUAD || nb == 0))
            LAL_TRY(lal::finish_partials(c, 1, a.ex.post));
        if(nb == 0)
            return LAL_OK;
        if(by == BY_LIST)
            launch_list<T, MODE>(c, a, nb);
        else if(by == BY_QUAD)
            c16 ? launch_quad<T, MODE, true>(c, a, nb) : launch_quad<T, MODE, false>(c, a, nb);
        else if(by == BY_NNZ)
        {
            auto* fn = c16 ? quad_nnz_kernel<T, MODE, true> : quad_nnz_kernel<T, MODE, false>;
            fn<<<nb, SPMV_THREADS, RP_LDS_BYTES + sizeof(T) * a.win, c->stream>>>(
                a.m, a.nnz, a.blocks, nb, a.win, a.rp, a.ci, a.c16, a.cbase, (const T*)a.val,
                (const T*)a.x, (const T*)a.d, (const T*)a.b, (T)a.alpha, (T)a.beta, (T*)a.y,
                (T*)a.r);
        }
        else
            staged_kernel<T, MODE><<<nb, SPMV_THREADS, 0, c->stream>>>(
                a.m, a.blocks, nb, a.rp, a.ci, (const T*)a.val, (const T*)a.x, (const T*)a.d,
                (const T*)a.b, (T)a.alpha, (T)a.beta, (T*)a.y, (T*)a.r);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    // (rowvec_can_dot holds)
    template <typename T>
    int launch_dot(lal_context* c, int mode, const lal::rv_args& a)
    {
        if(mode == lal::RV_ADD_DOT)
            launch_list<T, lal::RV_ADD_DOT>(c, a, a.nb);
        else if(mode == lal::RV_STEP_DOT && a.c16 && a.cbase)
            launch_quad<T, lal::RV_STEP_DOT, true>(c, a, a.nb);
        else if(mode == lal::RV_STEP_DOT)
            launch_quad<T, lal::RV_STEP_DOT, false>(c, a, a.nb);
        else if(a.c16 && a.cbase)
            launch_quad<T, lal::RV_SPMV_DOT, true>(c, a, a.nb);
        else
            launch_quad<T, lal::RV_SPMV_DOT, false>(c, a, a.nb);
        LAL_LAUNCHED();
        return LAL_OK;
    }
}

namespace lal
{
    bool rowvec_can_dot(int mode, const rv_args& a)
    {
        return a.blocks && a.nb > 0 && a.nb <= PCG_PARTS &&
               route(a) == (mode == RV_ADD_DOT ? BY_LIST : BY_QUAD);
    }

    template <typename T>
    int rowvec_launch(lal_context* c, int mode, const rv_args& a)
    {
        // what the mode's kernels gather
        LAL_REQUIRE(a.nnz == 0 || (mode == RV_JACOBI0 ? a.b && a.d : a.x != nullptr));
        switch(mode)
        {
        case RV_SPMV: return launch<T, RV_SPMV>(c, a);
        case RV_RESTRICT: return launch<T, RV_RESTRICT>(c, a);
        case RV_RESIDUAL: return launch<T, RV_RESIDUAL>(c, a);
        case RV_JACOBI: return launch<T, RV_JACOBI>(c, a);
        case RV_SMOOTHED: return launch<T, RV_SMOOTHED>(c, a);
        case RV_ADD: return launch<T, RV_ADD>(c, a);
        case RV_SPMV_DOT:
        case RV_ADD_DOT:
        case RV_STEP_DOT:
            LAL_REQUIRE(rowvec_can_dot(mode, a) && a.ex.part != nullptr &&
                        (mode == RV_STEP_DOT ? a.ex.gamma_part != nullptr : a.ex.w != nullptr));
            return launch_dot<T>(c, mode, a);
        default: return launch<T, RV_JACOBI0>(c, a);
        }
    }

    template int rowvec_launch<double>(lal_context*, int, const rv_args&);
    template int rowvec_launch<float>(lal_context*, int, const rv_args&);
}
