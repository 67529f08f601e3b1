// Block reductions of the PCG kernels: fixed orders, no atomics.
#pragma once

#include "lal_spmv.h"

namespace lal
{
    // A PCG reduction's last step: `part`'s partials into *slot (device) and,
    // when given, into *host_val and then *host_seq (mapped pinned memory) =
    // ++*counter (device).  part null: nothing to do.
    struct post_args
    {
        const double* part     = nullptr;
        int           count    = 0;
        double*       slot     = nullptr;
        double*       host_val = nullptr;
        unsigned*     host_seq = nullptr;
        unsigned*     counter  = nullptr;
    };

    // OP 0: sum; OP 1: maximum that keeps a NaN from either side, so that a
    // NaN anywhere in a vector reaches the solver's norm (and stops it)
    // whatever the order of the combination.
    template <int OP>
    __device__ __forceinline__ double combine(double a, double b)
    {
        return OP == 0 ? a + b : ((a != a || b < a) ? a : b);
    }

    // Block total of one value per lane (all lanes receive it).
    template <int OP>
    __device__ __forceinline__ double block_total(double v)
    {
        __shared__ double sh[SPMV_THREADS / 64];
        v = OP == 0 ? wave_sum(v) : wave_max_nan(v);
        __syncthreads();
        if((threadIdx.x & 63) == 0)
            sh[threadIdx.x >> 6] = v;
        __syncthreads();
        double t = sh[0];
#pragma unroll
        for(int w = 1; w < SPMV_THREADS / 64; w++)
            t = combine<OP>(t, sh[w]);
        return t;
    }

    // Total of a reduction's `count` partials, identical in every block; four
    // loads in flight per lane.
    template <int OP>
    __device__ __forceinline__ double total_of(const double* __restrict__ part, int count)
    {
        double v = 0.0;
        int    k = threadIdx.x;
        for(; k + 3 * SPMV_THREADS < count; k += 4 * SPMV_THREADS)
        {
            double p[4];
#pragma unroll
            for(int u = 0; u < 4; u++)
                p[u] = part[k + u * SPMV_THREADS];
#pragma unroll
            for(int u = 0; u < 4; u++)
                v = combine<OP>(v, p[u]);
        }
        for(; k < count; k += SPMV_THREADS)
            v = combine<OP>(v, part[k]);
        return block_total<OP>(v);
    }

    // One block: a.part into a.slot and the host's note.
    template <int OP>
    __device__ __forceinline__ void post_block(const post_args& a)
    {
        const double t = total_of<OP>(a.part, a.count);
        if(threadIdx.x == 0)
        {
            *a.slot = t;
            if(a.host_val)
            {
                const unsigned seq = *a.counter + 1;
                *a.counter         = seq;
                __hip_atomic_store(a.host_val, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                __hip_atomic_store(a.host_seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
    }
}
