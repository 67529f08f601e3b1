// The small end of the V-cycle as one dense operator.
//
// The last levels of a hierarchy hold a few thousand nonzeros: launched level
// by level (residual, restriction, ..., corrections back up) their kernels are
// pure latency, 3 to 4 us each, and one workgroup that walked them all out of
// LDS took 8 us of barriers.  But a V-cycle from zero with fixed sweeps is a
// linear map of its right-hand side, and with one pre- and one post-sweep
// (iterative_solvers/amg/amg.cpp:144-267, n1 = n2 = 1)
//
//     x = D^-1 b,  r = b - A x,  b_c = R r,  e = M_c b_c,
//     result = x + D^-1 r + Q e,   Q = P - D^-1 A P,
//
// so the level's map is
//
//     M = D^-1 (2 I - A D^-1) + Q M_c S,   S = R (I - A D^-1).
//
// The setup forms it in FP64, from the coarsest level's inverse up to the
// first level of at most CYCLE_ROWS rows, three launches a level; the cycle
// applies it as one matrix-vector product.
#include "lal_coarse.h"

namespace
{
    __device__ __forceinline__ void lds_add(double* p, double v)
    {
        (void)__hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    // S(k, :) = R(k, :) (I - A D^-1), a workgroup per row.  Each wavefront takes
    // every fourth entry of R's row and sums in LDS of its own: a wavefront's LDS
    // adds keep their order and the four sums are added in theirs, so the result
    // does not depend on timing.  Bound by the chain of A's rows, of which a
    // wavefront has four in flight; one wavefront per row took 90 us over the
    // levels of 552, 84 and 12 rows of a 25^3 diffusion hierarchy, this 39 us.
    __global__ void __launch_bounds__(256)
        restrict_rows_kernel(lal::cycle_level L, double* __restrict__ S)
    {
        __shared__ double sums[4][lal::CYCLE_ROWS];
        const int k = (int)blockIdx.x, lane = (int)threadIdx.x & 63;
        const int wave = (int)threadIdx.x >> 6;
        double*   s = sums[wave];
        for(int i = lane; i < L.m; i += 64)
            s[i] = 0.0;
        __syncthreads();
        const int re = L.rrp[k + 1];
        for(int base = L.rrp[k]; base < re; base += 256)
        {
            const int    e  = base + 4 * lane + wave;
            const bool   on = e < re;
            const int    j  = on ? L.rci[e] : 0;
            const double w  = on ? L.rv[e] : 0.0;
            const int    a0 = on ? L.arp[j] : 0, a1 = on ? L.arp[j + 1] : 0;
            if(on)
                lds_add(&s[j], w);
            const int n = min(64, (re - base + 3) >> 2);
            for(int u0 = 0; u0 < n; u0 += 4)
            {
                int    at[4], end[4], col[4];
                double wu[4], val[4];
#pragma unroll
                for(int u = 0; u < 4; u++)
                {
                    // (lanes past the row hold an empty range)
                    at[u]  = __shfl(a0, u0 + u, 64) + lane;
                    end[u] = __shfl(a1, u0 + u, 64);
                    wu[u]  = __shfl(w, u0 + u, 64);
                    col[u] = at[u] < end[u] ? L.aci[at[u]] : -1;
                    val[u] = at[u] < end[u] ? L.av[at[u]] : 0.0;
                }
#pragma unroll
                for(int u = 0; u < 4; u++)
                    if(col[u] >= 0)
                        val[u] *= L.dinv[col[u]];
#pragma unroll
                for(int u = 0; u < 4; u++)
                {
                    if(col[u] >= 0)
                        lds_add(&s[col[u]], -wu[u] * val[u]);
                    for(int t = at[u] + 64; t < end[u]; t += 64)
                        lds_add(&s[L.aci[t]], -wu[u] * (L.av[t] * L.dinv[L.aci[t]]));
                }
            }
        }
        __syncthreads();
        const int ld = lal::cycle_ld(L.m);
        for(int i = (int)threadIdx.x; i < ld; i += 256)
            S[(size_t)k * ld + i] =
                i < L.m ? (sums[0][i] + sums[1][i]) + (sums[2][i] + sums[3][i]) : 0.0;
    }

    // U = Mc S (mc x mc times mc x n), or S / a11 for a 1x1 coarsest level;
    // 32 x 32 tiles, 2 x 2 of them per lane.
    __global__ void __launch_bounds__(256)
        coarse_product_kernel(int mc, int n, const double* __restrict__ Mc, int ldc,
                              const double* __restrict__ a11, const double* __restrict__ S,
                              double* __restrict__ U)
    {
        constexpr int TK = 16;
        __shared__ double sa[TK][33], sb[TK][33];
        const int tid = (int)threadIdx.x, tx = tid & 15, ty = tid >> 4;
        const int r0 = blockIdx.y * 32, c0 = blockIdx.x * 32;
        double    acc[2][2] = {};
        if(Mc)
            for(int k0 = 0; k0 < mc; k0 += TK)
            {
#pragma unroll
                for(int h = 0; h < 2; h++)
                {
                    const int i = tid + 256 * h;
                    const int ar = r0 + (i >> 4), ak = k0 + (i & 15);
                    const int bk = k0 + (i >> 5), bc = c0 + (i & 31);
                    sa[i & 15][i >> 4] = ar < mc && ak < mc ? Mc[(size_t)ar * ldc + ak] : 0.0;
                    sb[i >> 5][i & 31] = bk < mc && bc < n ? S[(size_t)bk * n + bc] : 0.0;
                }
                __syncthreads();
#pragma unroll
                for(int k = 0; k < TK; k++)
                {
                    const double p0 = sa[k][ty], p1 = sa[k][ty + 16];
                    const double q0 = sb[k][tx], q1 = sb[k][tx + 16];
                    acc[0][0] = fma(p0, q0, acc[0][0]);
                    acc[0][1] = fma(p0, q1, acc[0][1]);
                    acc[1][0] = fma(p1, q0, acc[1][0]);
                    acc[1][1] = fma(p1, q1, acc[1][1]);
                }
                __syncthreads();
            }
#pragma unroll
        for(int a = 0; a < 2; a++)
#pragma unroll
            for(int b = 0; b < 2; b++)
            {
                const int row = r0 + ty + 16 * a, col = c0 + tx + 16 * b;
                if(row < mc && col < n)
                    U[(size_t)row * n + col] =
                        Mc ? acc[a][b] : S[(size_t)row * n + col] / a11[0];
            }
    }

    // M(i, :) = D^-1 (2 I - A D^-1)(i, :) + Q(i, :) U, a workgroup per row with up
    // to four columns per lane.  Bound by the L2: every entry of Q reads a row
    // of U.
    __global__ void __launch_bounds__(256)
        cycle_rows_kernel(lal::cycle_level L, const double* __restrict__ U,
                          double* __restrict__ M)
    {
        __shared__ double s[lal::CYCLE_ROWS];
        constexpr int     C  = lal::CYCLE_ROWS / 256;
        const int         i = (int)blockIdx.x, tid = (int)threadIdx.x;
        const int         ld = lal::cycle_ld(L.m);
        const double      di = L.dinv[i];
        for(int c = tid; c < L.m; c += 256)
            s[c] = 0.0;
        __syncthreads();
        for(int t = L.arp[i] + tid; t < L.arp[i + 1]; t += 256)
            lds_add(&s[L.aci[t]], -di * (L.av[t] * L.dinv[L.aci[t]]));
        if(tid == 0)
            lds_add(&s[i], 2.0 * di);
        double acc[C] = {};
#pragma unroll 4
        for(int t = L.qrp[i]; t < L.qrp[i + 1]; t++)
        {
            const double  w   = L.qv[t];
            const double* row = U + (size_t)L.qci[t] * ld;
#pragma unroll
            for(int u = 0; u < C; u++)
                if(tid + 256 * u < L.m)
                    acc[u] = fma(w, row[tid + 256 * u], acc[u]);
        }
        __syncthreads();
#pragma unroll
        for(int u = 0; u < C; u++)
        {
            const int c = tid + 256 * u;
            if(c < ld)
                M[(size_t)i * ld + c] = c < L.m ? s[c] + acc[u] : 0.0;
        }
    }

    // x = M b, a wavefront per row: 16 bytes of M per lane and load, eight loads
    // in flight, FP64 sums in either precision.  Bound by latency: 2.6 us at 496
    // rows and 4.3 us at 1000 (8 MB, 1 MB in each XCD's L2), where the residual,
    // the restriction, the LDS tail of the levels below and the correction took
    // 3.4 + 3.4 + 8.1 + 3.3 us.
    template <typename T>
    __global__ void __launch_bounds__(256)
        cycle_apply_kernel(int m, const double* __restrict__ M, const T* __restrict__ b,
                           T* __restrict__ x)
    {
        typedef double double2v __attribute__((ext_vector_type(2)));
        constexpr int C    = lal::CYCLE_ROWS / 128;
        const int     lane = (int)threadIdx.x & 63;
        const int     row  = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
        if(row >= m)
            return;
        const double2v* a = reinterpret_cast<const double2v*>(M + (size_t)row * lal::cycle_ld(m));
        double2v        v[C];
        double          p[C], q[C];
#pragma unroll
        for(int u = 0; u < C; u++)
        {
            const int c = 2 * (lane + 64 * u);
            v[u]        = c < m ? a[c >> 1] : double2v{0.0, 0.0};
            p[u]        = c < m ? (double)b[c] : 0.0;
            q[u]        = c + 1 < m ? (double)b[c + 1] : 0.0;
        }
        double s0 = 0.0, s1 = 0.0;
#pragma unroll
        for(int u = 0; u < C; u++)
        {
            s0 = fma(v[u].x, p[u], s0);
            s1 = fma(v[u].y, q[u], s1);
        }
        s0 += s1;
#pragma unroll
        for(int d = 32; d > 0; d >>= 1)
            s0 += __shfl_xor(s0, d, 64);
        if(lane == 0)
            x[row] = (T)s0;
    }
}

namespace lal
{
    int cycle_matrix(lal_context* c, const cycle_level& L, const double* Mc, int ldc,
                     const double* a11, double* S, double* U, double* M)
    {
        LAL_REQUIRE(L.m >= 1 && L.m <= CYCLE_ROWS && L.mc >= 1 && L.mc <= CYCLE_ROWS);
        LAL_REQUIRE(Mc != nullptr || (L.mc == 1 && a11 != nullptr));
        const int ld = cycle_ld(L.m);
        restrict_rows_kernel<<<L.mc, 256, 0, c->stream>>>(L, S);
        LAL_LAUNCHED();
        coarse_product_kernel<<<dim3((ld + 31) / 32, (L.mc + 31) / 32), 256, 0, c->stream>>>(
            L.mc, ld, Mc, ldc, a11, S, U);
        LAL_LAUNCHED();
        cycle_rows_kernel<<<L.m, 256, 0, c->stream>>>(L, U, M);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    template <typename T>
    int cycle_apply(lal_context* c, int m, const double* M, const T* b, T* x)
    {
        LAL_REQUIRE(m >= 1 && m <= CYCLE_ROWS && (reinterpret_cast<uintptr_t>(M) & 15) == 0);
        cycle_apply_kernel<T><<<(m + 3) / 4, 256, 0, c->stream>>>(m, M, b, x);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    template int cycle_apply<double>(lal_context*, int, const double*, const double*, double*);
    template int cycle_apply<float>(lal_context*, int, const double*, const float*, float*);
}
