// CSR SpMV, residual and diagonal extraction for gfx950.
//
// y = alpha*A*x + beta*y follows backend/host/host_matrix_vector.cpp:59-84
// (row sum s = fma(val, x[col], s), then beta == 0 ? alpha*s :
// fma(alpha, s, beta*y)); r = b - A*x follows :35-57 (s += val*x, two
// roundings).  The row-block layout and LDS staging are described in
// lal_spmv.h.
#include "lal_rowvec.h"

#include <algorithm>
#include <climits>

#include <vector>

namespace
{
    using lal::SPMV_THREADS;

    // MODE 0: y = alpha*A*x + beta*y ;  MODE 1: y = b - A*x
    template <typename T, typename ACC, int MODE>
    __global__ void __launch_bounds__(SPMV_THREADS)
        csrmv_kernel(const int* __restrict__ blocks, int nb, int m, const int* __restrict__ rp,
                     const int* __restrict__ ci, const T* __restrict__ val,
                     const T* __restrict__ x, ACC alpha, ACC beta, const T* __restrict__ b,
                     T* __restrict__ y, int exact)
    {
        constexpr int CAP = lal::spmv_cap<T>::value;
        __shared__ T  s_v[CAP];
        __shared__ T  s_x[CAP];
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
        const int  rs     = active ? s_rp[lrow] : 0;
        const int  re     = active ? s_rp[lrow + 1] : 0;

        ACC acc = 0;
        for(int cs = base; cs < end; cs += CAP)
        {
            const int len = min(CAP, end - cs);
#pragma unroll 4
            for(int k = tid; k < len; k += SPMV_THREADS)
            {
                int c  = ci[cs + k];
                s_v[k] = val[cs + k];
                s_x[k] = x[c];
            }
            __syncthreads();
            if(active)
            {
                const int a = max(rs, cs) - cs;
                const int e = min(re, cs + len) - cs;
                for(int j = a + lig; j < e; j += g)
                {
                    if(MODE == 0)
                        acc = fma((ACC)s_v[j], (ACC)s_x[j], acc);
                    else
                        acc = acc + (ACC)s_v[j] * (ACC)s_x[j];
                }
            }
            __syncthreads();
        }
        if(g > 1)
            acc = lal::group_sum(acc, g);
        if(active && lig == 0)
        {
            const int row = r0 + lrow;
            if(MODE == 0)
                y[row] = (T)(beta == (ACC)0 ? alpha * acc : fma(alpha, acc, beta * (ACC)y[row]));
            else
                y[row] = (T)((ACC)b[row] - acc);
        }
    }

    // Sets `bit` in *bad if a column index lies outside [0, n): an invalid matrix
    // is refused before any gather can run off the end of x.
    __global__ void __launch_bounds__(256)
        check_cols_kernel(int nnz, int n, const int* __restrict__ ci, int* __restrict__ bad,
                          int bit = 1)
    {
        int k = blockIdx.x * 256 + threadIdx.x;
        int stride = gridDim.x * 256;
        int b = 0;
        for(; k < nnz; k += stride)
            b |= (unsigned)ci[k] >= (unsigned)n;
        if(__any(b) && (threadIdx.x & 63) == 0)
            atomicOr(bad, bit);
    }

    __global__ void __launch_bounds__(256)
        diagonal_kernel(int m, const int* __restrict__ rp, const int* __restrict__ ci,
                        const double* __restrict__ val, double* __restrict__ d)
    {
        int i = blockIdx.x * 256 + threadIdx.x;
        if(i >= m)
            return;
        for(int j = rp[i]; j < rp[i + 1]; j++)
            if(ci[j] == i)
            {
                d[i] = val[j];
                break;
            }
    }

    // ------------------------------------------------------ row-block analysis
    // Rows are packed greedily: a block closes at 256 rows or when the next
    // row would push it past `cap` nonzeros; a row longer than cap is a block of
    // its own.  The packing starts anew every RB_TILE rows, so that a workgroup
    // packs each tile by itself: all rows' "next block" are found at once in
    // LDS (a binary search in the staged row pointer) and one lane follows
    // them.  Several operators share a launch (a hierarchy analyses all of its
    // own at once, without a copy of a row pointer to the host).
    constexpr int LIST_CAP = 2044; // nonzeros of a block with a column list
    constexpr int RB_TILE  = 2048;
    constexpr int RB_BATCH = 24; // operators per launch (their table is a kernel argument)

    // (a descriptor's own analysis has one: a launch copies its arguments)
    template <int MAX>
    struct rb_table
    {
        int        n;
        lal::rb_op op[MAX];
    };

    // results of one operator, in the order read back
    enum
    {
        RB_NBLOCKS = 0,
        RB_WIN     = 1, // widest 4-aligned nonzero window of a block (<= 2052)
        RB_BAD     = 2, // 1: row pointer not from 0 to nnz, 2: not monotone, 4: column range
        RB_WIDE    = 3, // a block spans more than 65535 columns
        RB_LMAX    = 4, // longest list of distinct columns of a block
        RB_LONG    = 5, // a block of more than LIST_CAP nonzeros (one long row) or 131072 columns
        RB_FAR     = 6, // a list reaches beyond 65536 columns
        RB_RES     = 7
    };

    // Position of `at` among the operators' starts (ascending).
    template <int MAX, typename F>
    __device__ __forceinline__ int rb_find(const rb_table<MAX>& t, int at, F start)
    {
        int k = 0;
        while(k + 1 < t.n && start(t.op[k + 1]) <= at)
            k++;
        return k;
    }

    // Tiles of one operator that the second pass scans by itself.
    constexpr int RB_SCAN = 256;

    // WRITE false: blocks per tile into tcount, the widest window and the row
    // pointer's faults into res.  WRITE true: the block table, at the tile's
    // offset that the scan left in tcount; with `scan` (one operator of at most
    // RB_SCAN tiles) every workgroup adds up the counts before its own.
    template <bool WRITE, int MAX>
    __global__ void __launch_bounds__(256)
        rb_tile_kernel(rb_table<MAX> tab, int* __restrict__ tcount, int* __restrict__ res, bool scan)
    {
        __shared__ int            s_rp[RB_TILE + 1];
        __shared__ unsigned short s_next[RB_TILE];
        __shared__ int            s_n, s_sum[2][4];
        const int    k   = rb_find(tab, (int)blockIdx.x, [](const lal::rb_op& o) { return o.tile0; });
        const lal::rb_op o = tab.op[k];
        int*         out = res + RB_RES * k;
        const int    tid = (int)threadIdx.x;
        int          all = 0, at = 0; // blocks of the operator, and before this tile
        if(WRITE && scan)
        {
            const int v = tid < o.ntiles ? tcount[tid] : 0;
            const int a = lal::wave_sum(v), b = lal::wave_sum(tid < (int)blockIdx.x ? v : 0);
            if((tid & 63) == 0)
            {
                s_sum[0][tid >> 6] = a;
                s_sum[1][tid >> 6] = b;
            }
            __syncthreads();
            for(int w = 0; w < 4; w++)
            {
                all += s_sum[0][w];
                at += s_sum[1][w];
            }
            if(blockIdx.x == 0 && tid == 0)
                out[RB_NBLOCKS] = all;
        }
        else if(WRITE)
        {
            all = out[RB_NBLOCKS];
            at  = tcount[blockIdx.x];
        }
        if(WRITE && (out[RB_BAD] != 0 || all > o.ub))
            return;
        const int r0  = ((int)blockIdx.x - o.tile0) * RB_TILE;
        const int n   = min(RB_TILE, o.m - r0);
        for(int i = tid; i <= n; i += 256)
            s_rp[i] = o.rp[r0 + i];
        __syncthreads();
        if(!WRITE)
        {
            int bad = 0;
            for(int i = tid; i < n; i += 256)
                bad |= s_rp[i + 1] < s_rp[i] ? 2 : 0;
            if(tid == 0)
                bad |= (r0 == 0 && s_rp[0] != 0) || (r0 + n == o.m && s_rp[n] != o.nnz) ? 1 : 0;
            if(bad)
                atomicOr(out + RB_BAD, bad);
        }
        // the block from row i ends before the first row t (at most 256 on)
        // with rp[t + 1] - rp[i] > cap
        for(int i = tid; i < n; i += 256)
        {
            const long long top = (long long)s_rp[i] + o.cap;
            int             lo = i, hi = min(n, i + SPMV_THREADS); // rp[lo] <= top
            while(lo < hi)
            {
                const int mid = (lo + hi + 1) >> 1;
                if(s_rp[mid] <= top)
                    lo = mid;
                else
                    hi = mid - 1;
            }
            s_next[i] = (unsigned short)max(lo, i + 1);
        }
        __syncthreads();
        if(tid == 0)
        {
            // reached rows are read once: the list of block starts replaces the
            // links behind the walk
            int cnt = 0;
            for(int r = 0; r < n;)
            {
                const int next = s_next[r];
                s_next[cnt++]  = (unsigned short)r;
                r              = next;
            }
            s_n = cnt;
        }
        __syncthreads();
        const int nb = s_n;
        if(!WRITE)
        {
            int win = 4;
            for(int b = tid; b < nb; b += 256)
            {
                const int i = s_next[b], e = b + 1 < nb ? (int)s_next[b + 1] : n;
                win         = max(win, min(((s_rp[e] + 3) & ~3) - (s_rp[i] & ~3), 2052));
            }
            win = lal::wave_max(win);
            if((tid & 63) == 0 && win > 4)
                atomicMax(out + RB_WIN, win);
            if(tid == 0)
                tcount[blockIdx.x] = nb;
            return;
        }
        int*      meta = o.blocks + lal::block_meta_offset(all);
        for(int b = tid; b < nb; b += 256)
        {
            const int i = s_next[b], e = b + 1 < nb ? (int)s_next[b + 1] : n;
            o.blocks[at + b]           = r0 + i;
            meta[4 * (size_t)(at + b)]     = r0 + i;
            meta[4 * (size_t)(at + b) + 1] = r0 + e;
            meta[4 * (size_t)(at + b) + 2] = s_rp[i];
            meta[4 * (size_t)(at + b) + 3] = s_rp[e];
        }
        if(tid == 0 && r0 + n == o.m)
            o.blocks[all] = o.m;
    }

    // One workgroup per operator: its tiles' block counts become offsets.
    template <int MAX>
    __global__ void __launch_bounds__(256)
        rb_scan_kernel(rb_table<MAX> tab, int* __restrict__ tcount, int* __restrict__ res)
    {
        __shared__ int  s_w[4];
        const int       k    = (int)blockIdx.x;
        const lal::rb_op o   = tab.op[k];
        const int       lane = (int)threadIdx.x & 63, wid = (int)threadIdx.x >> 6;
        int             carry = 0;
        for(int t0 = 0; t0 < o.ntiles; t0 += 256)
        {
            const int i   = t0 + (int)threadIdx.x;
            const int v   = i < o.ntiles ? tcount[o.tile0 + i] : 0;
            int       inc = v;
#pragma unroll
            for(int d = 1; d < 64; d <<= 1)
            {
                const int q = __shfl_up(inc, d, 64);
                inc += lane >= d ? q : 0;
            }
            if(lane == 63)
                s_w[wid] = inc;
            __syncthreads();
            int off = carry, tot = 0;
            for(int w = 0; w < 4; w++)
            {
                off += w < wid ? s_w[w] : 0;
                tot += s_w[w];
            }
            if(i < o.ntiles)
                tcount[o.tile0 + i] = off + inc - v;
            carry += tot;
            __syncthreads();
        }
        if(threadIdx.x == 0)
            res[RB_RES * k + RB_NBLOCKS] = carry;
    }

    // Four 16-bit values for entries e..e+3 (e a multiple of 4) of dst, those in
    // [e0, e1) only: the quad at either end is shared with the next block.
    __device__ __forceinline__ void store_quad16(unsigned short* __restrict__ dst, int e, int e0,
                                                 int e1, const unsigned (&x)[4])
    {
        if(e >= e0 && e + 4 <= e1)
            *reinterpret_cast<uint2*>(dst + e) = {x[0] | x[1] << 16, x[2] | x[3] << 16};
        else
#pragma unroll
            for(int j = 0; j < 4; j++)
                if(e + j >= e0 && e + j < e1)
                    dst[e + j] = (unsigned short)x[j];
    }

    // One workgroup per row block (the grid holds every operator's largest
    // possible number of blocks): the block's column range, its base (the
    // smallest column) and every entry's offset from it as 16 bits; RB_WIDE is
    // set when a block spans more than 65535 columns.  Where asked for, also the
    // block's distinct columns: a bitmap of the span in LDS, whose running
    // population count is each column's place in the ascending list.
    // Every lane holds its two quads of columns in registers from the first read
    // on (reading them again for each of the four passes, a two-byte store per
    // entry and one lane unpacking a bitmap word took 770 us over the operators
    // of a 121^3 diffusion hierarchy; now 460 us, bound by the chain of
    // barriers).
    template <int MAX>
    __global__ void __launch_bounds__(256)
        rb_columns_kernel(rb_table<MAX> tab, int* __restrict__ res)
    {
        typedef int            int4v __attribute__((ext_vector_type(4)));
        typedef unsigned       uint4v __attribute__((ext_vector_type(4)));
        typedef unsigned short ushort4v __attribute__((ext_vector_type(4)));
        __shared__ uint4v   s_bits4[1024];
        __shared__ ushort4v s_place4[1024];
        __shared__ unsigned s_list2[(LIST_CAP + 4) / 2];
        __shared__ int      s_w[2][4];
        __shared__ int      sh_mn[4], sh_mx[4];
        unsigned* const       s_bits  = reinterpret_cast<unsigned*>(s_bits4);
        unsigned short* const s_place = reinterpret_cast<unsigned short*>(s_place4);
        unsigned short* const s_list  = reinterpret_cast<unsigned short*>(s_list2);
        const int k = rb_find(tab, (int)blockIdx.x, [](const lal::rb_op& o) { return o.blk0; });
        const lal::rb_op o   = tab.op[k];
        int*             out = res + RB_RES * k;
        const int        nb  = out[RB_NBLOCKS];
        const int        b   = (int)blockIdx.x - o.blk0;
        if(o.c16 == nullptr || out[RB_BAD] != 0 || nb > o.ub || b >= nb)
            return;
        const int4v mt = reinterpret_cast<const int4v*>(o.blocks + lal::block_meta_offset(nb))[b];
        const int   e0 = mt.z, e1 = mt.w, tid = (int)threadIdx.x;
        const int   q0 = e0 & ~3;
        const bool  held = e1 - q0 <= 2048; // else: one long row, or an unlucky 2048
        const bool  al   = ((size_t)o.ci & 15) == 0;
        int         col[2][4];
        int         mn = INT_MAX, mx = INT_MIN;
        if(held)
        {
#pragma unroll
            for(int h = 0; h < 2; h++)
            {
                const int e = q0 + 4 * (tid + 256 * h);
                if(al && e >= e0 && e + 4 <= e1)
                {
                    const int4v q = *reinterpret_cast<const int4v*>(o.ci + e);
                    col[h][0] = q.x, col[h][1] = q.y, col[h][2] = q.z, col[h][3] = q.w;
                }
                else
#pragma unroll
                    for(int j = 0; j < 4; j++)
                        col[h][j] = e + j >= e0 && e + j < e1 ? o.ci[e + j] : 0;
            }
#pragma unroll
            for(int h = 0; h < 2; h++)
#pragma unroll
                for(int j = 0; j < 4; j++)
                {
                    const int e = q0 + 4 * (tid + 256 * h) + j;
                    if(e >= e0 && e < e1)
                    {
                        mn = min(mn, col[h][j]);
                        mx = max(mx, col[h][j]);
                    }
                }
        }
        else
            for(int e = e0 + tid; e < e1; e += 256)
            {
                mn = min(mn, o.ci[e]);
                mx = max(mx, o.ci[e]);
            }
#pragma unroll
        for(int d = 32; d > 0; d >>= 1)
        {
            mn = min(mn, __shfl_xor(mn, d, 64));
            mx = max(mx, __shfl_xor(mx, d, 64));
        }
        const int lane = tid & 63, wid = tid >> 6;
        if(lane == 0)
        {
            sh_mn[wid] = mn;
            sh_mx[wid] = mx;
        }
        __syncthreads();
        mn = min(min(sh_mn[0], sh_mn[1]), min(sh_mn[2], sh_mn[3]));
        mx = max(max(sh_mx[0], sh_mx[1]), max(sh_mx[2], sh_mx[3]));
        const int       base = e1 > e0 ? mn : 0;
        const long long span = e1 > e0 ? (long long)mx - mn : 0;
        if(tid == 0)
        {
            o.cbase[b] = base;
            if(span > 65535)
                atomicOr(out + RB_WIDE, 1);
        }
        if(held)
        {
#pragma unroll
            for(int h = 0; h < 2; h++)
            {
                unsigned x[4];
#pragma unroll
                for(int j = 0; j < 4; j++)
                    x[j] = (unsigned)(col[h][j] - base) & 0xffffu;
                store_quad16(o.c16, q0 + 4 * (tid + 256 * h), e0, e1, x);
            }
        }
        else
            for(int e = e0 + tid; e < e1; e += 256)
                o.c16[e] = (unsigned short)(o.ci[e] - base);
        if(o.lpos == nullptr)
            return;
        if(e1 - e0 > LIST_CAP || span > 131071)
        {
            if(tid == 0)
                atomicOr(out + RB_LONG, 1);
            return;
        }
        const int words = e1 > e0 ? (int)(span >> 5) + 1 : 0; // at most 4096
        const int w4    = (words + 3) >> 2;
        for(int w = tid; w < w4; w += 256)
            s_bits4[w] = uint4v{0, 0, 0, 0};
        __syncthreads();
#pragma unroll
        for(int h = 0; h < 2; h++)
#pragma unroll
            for(int j = 0; j < 4; j++)
            {
                const int e = q0 + 4 * (tid + 256 * h) + j;
                const int off = col[h][j] - base;
                if(e >= e0 && e < e1)
                    atomicOr(&s_bits[off >> 5], 1u << (off & 31));
            }
        __syncthreads();
        int carry = 0, turn = 0;
        for(int w0 = 0; w0 < w4; w0 += 256, turn ^= 1)
        {
            const int    w    = w0 + tid;
            const uint4v bits = w < w4 ? s_bits4[w] : uint4v{0, 0, 0, 0};
            const int n0 = __popc(bits.x), n1 = n0 + __popc(bits.y), n2 = n1 + __popc(bits.z);
            const int n  = n2 + __popc(bits.w);
            int       inc = n;
#pragma unroll
            for(int d = 1; d < 64; d <<= 1)
            {
                const int q = __shfl_up(inc, d, 64);
                inc += lane >= d ? q : 0;
            }
            if(lane == 63)
                s_w[turn][wid] = inc;
            __syncthreads();
            int at = carry + inc - n;
#pragma unroll
            for(int v = 0; v < 4; v++)
            {
                at += v < wid ? s_w[turn][v] : 0;
                carry += s_w[turn][v];
            }
            if(w < w4)
                s_place4[w] = ushort4v{(unsigned short)at, (unsigned short)(at + n0),
                                       (unsigned short)(at + n1), (unsigned short)(at + n2)};
        }
        __syncthreads();
#pragma unroll
        for(int h = 0; h < 2; h++)
        {
            const int eq = q0 + 4 * (tid + 256 * h);
            unsigned  x[4];
#pragma unroll
            for(int j = 0; j < 4; j++)
            {
                x[j] = 0;
                if(eq + j >= e0 && eq + j < e1)
                {
                    const int      off  = col[h][j] - base;
                    const unsigned less = s_bits[off >> 5] & ((1u << (off & 31)) - 1u);
                    const int      at   = s_place[off >> 5] + __popc(less);
                    s_list[at]          = (unsigned short)off;
                    x[j]                = 4u * (unsigned)at;
                }
            }
            store_quad16(o.lpos, eq, e0, e1, x);
        }
        // the last quad is read whole
        if(b == nb - 1 && tid < (-o.nnz & 3))
            o.lpos[o.nnz + tid] = 0;
        if(tid == 0)
        {
            if(carry & 1)
                s_list[carry] = (unsigned short)span; // (its low 16 bits)
            // (words from 2048 on start the offsets of 65536 and more)
            const int near     = words > 2048 ? s_place[2048] : carry;
            const int split    = lal::list_split(carry, near);
            o.lmeta[2 * b]     = carry | split << 12 | lal::spmv_group_log(mt.y - mt.x) << 24;
            o.lmeta[2 * b + 1] = base;
            // (one address for all blocks: few of them raise it)
            if(carry > *(volatile int*)(out + RB_LMAX))
                atomicMax(out + RB_LMAX, carry);
            if(near < carry && *(volatile int*)(out + RB_FAR) == 0)
                atomicOr(out + RB_FAR, 1);
        }
        __syncthreads();
        unsigned* const list = reinterpret_cast<unsigned*>(o.list + lal::list_start(e0, b));
        for(int i = tid; i < (carry + 1) >> 1; i += 256)
            list[i] = s_list2[i];
    }

    template <typename T, typename ACC, int MODE>
    int csrmv_launch(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz, ACC alpha,
                     const int* rp, const int* ci, const T* v, const T* x, ACC beta,
                     const T* b, T* y)
    {
        LAL_REQUIRE(c != nullptr && m >= 0 && n >= 0 && nnz >= 0);
        if(m == 0)
            return LAL_OK;
        LAL_REQUIRE(rp != nullptr && y != nullptr);
        LAL_REQUIRE(nnz == 0 || (ci != nullptr && v != nullptr && x != nullptr));
        if(d)
            LAL_REQUIRE(d->m == m && d->nnz == nnz);
        if(d && !d->exact)
        {
            lal::rv_args a{m,    d->nnz, d->by_nnz, d->d_blocks, d->nblocks,     rp,           ci, v, x, nullptr,
                           b,    y,           nullptr,        (double)alpha, (double)beta, d->win};
            a.keep = d->keep;
            lal::use_c16(a, d);
            return lal::rowvec_launch<T>(c, MODE == 0 ? lal::RV_SPMV : lal::RV_RESIDUAL, a);
        }
        // an exact descriptor, or none: one lane per row in CSR order (the
        // host loop's rounding)
        int nb = lal::spmv_grid(d, m);
        csrmv_kernel<T, ACC, MODE><<<nb, SPMV_THREADS, 0, c->stream>>>(
            d ? d->d_blocks : nullptr, nb, m, rp, ci, v, x, alpha, beta, b, y, 1);
        LAL_LAUNCHED();
        return LAL_OK;
    }
}

namespace lal
{
    int raise_bad_columns(lal_context* c, int nnz, int n, const int* ci, int* flag)
    {
        if(nnz == 0)
            return LAL_OK;
        check_cols_kernel<<<grid_for(nnz, 256, 4096), 256, 0, c->stream>>>(nnz, n, ci, flag);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    // Nonzeros per row block: 2048 (the kernels' LDS chunk) for large
    // matrices; for small ones it shrinks, down to 256, so that a launch still
    // has about 1024 workgroups: their time is one latency chain per
    // workgroup, and more, shorter chains spread over all CUs finish sooner.
    // With column lists a larger block also reads fewer columns of x per
    // nonzero, and one workgroup per CU is enough (gradient on 64^3, whose
    // second level holds 1.2 million nonzeros: 1024 workgroups 15.7 ms, 512
    // 15.4, 256 15.2; 4096 17.6).
    static int block_cap(int nnz, bool lists)
    {
        int cap = lists ? LIST_CAP : spmv_cap<double>::value;
        while(cap > 256 && nnz / (lists ? 256 : 1024) < cap)
            cap >>= 1;
        return cap;
    }

    // Requests [first, ...) in one pass, MAX of them at most.
    template <int MAX>
    static int analyse_some(lal_context* c, const std::vector<rb_request>& req, size_t first,
                            arena* mem, arena* tmp)
    {
        temps         t(c, tmp);
        rb_table<MAX> tab{};
        int           tiles = 0, blocks = 0;
        tab.n               = (int)std::min(req.size() - first, (size_t)MAX);
        for(int k = 0; k < tab.n; k++)
        {
            const rb_request& q = req[first + k];
            rb_op&            o = tab.op[k];
            o.rp     = q.rp;
            o.ci     = q.ci;
            o.m      = q.m;
            o.nnz    = q.nnz;
            // (the list kernel takes a block as 512 quads of four)
            o.cap    = block_cap(q.nnz, q.want_list);
            o.tile0  = tiles;
            o.ntiles = std::max((q.m + RB_TILE - 1) / RB_TILE, 1);
            o.blk0   = blocks;
            // a block that is neither of 256 rows nor a tile's last holds
            // more than cap nonzeros together with its successor
            o.ub = q.m / SPMV_THREADS + (int)(2LL * q.nnz / o.cap) + o.ntiles + 1;
            tiles += o.ntiles;
            blocks += o.ub;
            LAL_TRY(q.d->arrays(mem, o.ub));
            o.blocks = q.d->d_blocks;
            if(mem && q.want16 && q.nnz > 0)
            {
                // whole 16-byte lines: the kernels load four entries at a time
                LAL_TRY(mem->get(&q.d->d_c16, ((size_t)q.nnz + 7) & ~(size_t)7));
                LAL_TRY(mem->get(&q.d->d_cbase, o.ub));
                o.c16   = q.d->d_c16;
                o.cbase = q.d->d_cbase;
                if(q.want_list)
                {
                    LAL_TRY(mem->get(&q.d->d_lpos, ((size_t)q.nnz + 7) & ~(size_t)7));
                    LAL_TRY(mem->get(&q.d->d_list, list_start(q.nnz, o.ub) + 4));
                    LAL_TRY(mem->get(&q.d->d_lmeta, 2 * (size_t)o.ub));
                    o.lpos  = q.d->d_lpos;
                    o.list  = q.d->d_list;
                    o.lmeta = q.d->d_lmeta;
                }
            }
        }
        // A single operator of few tiles, as a caller's descriptor mostly is,
        // takes the context's flags (zero between calls) and reduction
        // workspace for its results and counts: no allocation, no clearing and
        // no scan of its own.  128^2 Poisson: 88 to 99 us without this and with a
        // table of 24 operators among the arguments, 40 so, 58 on the host; 5000
        // rows of up to 2500 entries 115, 55, 58; 100^3 (the general way) 89 and
        // 640 on the host.
        const bool few    = tab.n == 1 && tiles <= RB_SCAN;
        int *      tcount = nullptr, *res = nullptr;
        int        h[RB_RES * MAX] = {};
        static_assert(RB_RES <= LAL_FLAGS && RB_SCAN <= 2 * LAL_RED_BLOCKS);
        if(few)
        {
            res    = c->d_flag;
            tcount = reinterpret_cast<int*>(c->d_part);
        }
        else
        {
            LAL_TRY(t.get(&res, RB_RES * MAX));
            LAL_TRY(t.get(&tcount, tiles));
            LAL_TRY(lal_fill_i32(c, res, RB_RES * MAX, 0));
        }
        rb_tile_kernel<false, MAX><<<tiles, 256, 0, c->stream>>>(tab, tcount, res, few);
        LAL_LAUNCHED();
        if(!few)
        {
            rb_scan_kernel<MAX><<<tab.n, 256, 0, c->stream>>>(tab, tcount, res);
            LAL_LAUNCHED();
        }
        rb_tile_kernel<true, MAX><<<tiles, 256, 0, c->stream>>>(tab, tcount, res, few);
        LAL_LAUNCHED();
        if(mem)
        {
            rb_columns_kernel<MAX><<<blocks, 256, 0, c->stream>>>(tab, res);
            LAL_LAUNCHED();
        }
        for(int k = 0; k < tab.n; k++)
            if(req[first + k].check_n >= 0 && tab.op[k].nnz > 0)
            {
                check_cols_kernel<<<grid_for(tab.op[k].nnz, 256, 4096), 256, 0, c->stream>>>(
                    tab.op[k].nnz, req[first + k].check_n, tab.op[k].ci,
                    res + RB_RES * k + RB_BAD, 4);
                LAL_LAUNCHED();
            }
        LAL_TRY(read_ints(c, res, RB_RES * tab.n, h, few));
        for(int k = 0; k < tab.n; k++)
        {
            const rb_request& q = req[first + k];
            const int*        r = h + RB_RES * k;
            if(r[RB_BAD] & 4)
                set_last_error("column index outside [0, n)");
            else if(r[RB_BAD] & 1)
                set_last_error("row_ptr does not start at 0 or end at nnz");
            else if(r[RB_BAD] & 2 || r[RB_NBLOCKS] > tab.op[k].ub)
                set_last_error("row_ptr is not monotone");
            else
            {
                q.d->nblocks = r[RB_NBLOCKS];
                q.d->win     = std::max(r[RB_WIN], 4);
                if(r[RB_WIDE])
                    q.d->d_c16 = nullptr;
                if(q.d->d_lpos && !r[RB_LONG])
                {
                    q.d->list_max = r[RB_LMAX];
                    q.d->list_far = r[RB_FAR] != 0;
                }
                continue;
            }
            return LAL_ERR_INVALID;
        }
        return LAL_OK;
    }

    int analyse(lal_context* c, const std::vector<rb_request>& req, arena* mem, arena* tmp)
    {
        if(req.size() == 1)
            return analyse_some<1>(c, req, 0, mem, tmp);
        for(size_t first = 0; first < req.size(); first += RB_BATCH)
            LAL_TRY(analyse_some<RB_BATCH>(c, req, first, mem, tmp));
        return LAL_OK;
    }

    int csrmv_analysis_dev(lal_context* c, int m, int n, int nnz, const int* rp,
                           const int* ci, int exact, lal_csrmv_info** out)
    {
        auto* d   = new lal_csrmv_info;
        d->m      = m;
        d->nnz    = nnz;
        d->exact  = exact;
        d->by_nnz = m != n;
        const int st = analyse(c, {{d, rp, ci, m, nnz, false, n}}, nullptr, nullptr);
        if(st != LAL_OK)
        {
            lal_csrmv_descr_destroy(d);
            return st;
        }
        *out = d;
        return LAL_OK;
    }

    int csrmv_f64(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz, double alpha,
                  const int* rp, const int* ci, const double* v, const double* x, double beta,
                  double* y)
    {
        return csrmv_launch<double, double, 0>(c, d, m, n, nnz, alpha, rp, ci, v, x, beta,
                                               nullptr, y);
    }

    int csrmv_f32(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz, float alpha,
                  const int* rp, const int* ci, const float* v, const float* x, float beta,
                  float* y)
    {
        return csrmv_launch<float, float, 0>(c, d, m, n, nnz, alpha, rp, ci, v, x, beta,
                                             nullptr, y);
    }

    int residual_f64(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz,
                     const int* rp, const int* ci, const double* v, const double* x,
                     const double* b, double* r)
    {
        LAL_REQUIRE(m == 0 || b != nullptr);
        return csrmv_launch<double, double, 1>(c, d, m, n, nnz, 0.0, rp, ci, v, x, 0.0, b, r);
    }

    int residual_f32(lal_context* c, const lal_csrmv_info* d, int m, int n, int nnz,
                     const int* rp, const int* ci, const float* v, const float* x,
                     const float* b, float* r)
    {
        LAL_REQUIRE(m == 0 || b != nullptr);
        return csrmv_launch<float, float, 1>(c, d, m, n, nnz, 0.0f, rp, ci, v, x, 0.0f, b, r);
    }

    int diagonal_f64(lal_context* c, int m, const int* rp, const int* ci, const double* v,
                     double* d)
    {
        if(m == 0)
            return LAL_OK;
        diagonal_kernel<<<grid_for(m, 256), 256, 0, c->stream>>>(m, rp, ci, v, d);
        LAL_LAUNCHED();
        return LAL_OK;
    }
}

int lal_csrmv_info::arrays(lal::arena* mem, int nb)
{
    const size_t ints = lal::block_meta_offset(nb) + 4 * (size_t)nb;
    owned             = mem == nullptr;
    if(mem)
        return mem->get(&d_blocks, ints);
    return lal::device_malloc(reinterpret_cast<void**>(&d_blocks), sizeof(int) * ints);
}

extern "C" int lal_csrmv_analysis(lal_handle c, int m, int n, int nnz, const int* row_ptr,
                                  const int* col_ind, int exact, lal_csrmv_descr* descr)
{
    LAL_REQUIRE(c != nullptr && descr != nullptr && m >= 0 && n >= 0 && nnz >= 0);
    LAL_REQUIRE(row_ptr != nullptr && (nnz == 0 || col_ind != nullptr));
    *descr = nullptr;
    return lal::csrmv_analysis_dev(c, m, n, nnz, row_ptr, col_ind, exact, descr);
}

extern "C" int lal_csrmv_descr_destroy(lal_csrmv_descr d)
{
    if(!d)
        return LAL_OK;
    if(d->owned && d->d_blocks)
        (void)hipFree(d->d_blocks);
    delete d;
    return LAL_OK;
}

extern "C" int lal_csrmv_f64(lal_handle c, lal_csrmv_descr d, int m, int n, int nnz,
                             double alpha, const int* rp, const int* ci, const double* v,
                             const double* x, double beta, double* y)
{
    return lal::csrmv_f64(c, d, m, n, nnz, alpha, rp, ci, v, x, beta, y);
}

extern "C" int lal_csrmv_f32(lal_handle c, lal_csrmv_descr d, int m, int n, int nnz,
                             float alpha, const int* rp, const int* ci, const float* v,
                             const float* x, float beta, float* y)
{
    return lal::csrmv_f32(c, d, m, n, nnz, alpha, rp, ci, v, x, beta, y);
}

extern "C" int lal_residual_f64(lal_handle c, lal_csrmv_descr d, int m, int n, int nnz,
                                const int* rp, const int* ci, const double* v, const double* x,
                                const double* b, double* r)
{
    return lal::residual_f64(c, d, m, n, nnz, rp, ci, v, x, b, r);
}

extern "C" int lal_residual_f32(lal_handle c, lal_csrmv_descr d, int m, int n, int nnz,
                                const int* rp, const int* ci, const float* v, const float* x,
                                const float* b, float* r)
{
    return lal::residual_f32(c, d, m, n, nnz, rp, ci, v, x, b, r);
}

extern "C" int lal_diagonal_f64(lal_handle c, int m, const int* rp, const int* ci,
                                const double* v, double* d)
{
    LAL_REQUIRE(c != nullptr && m >= 0);
    LAL_REQUIRE(m == 0 || (rp != nullptr && d != nullptr));
    return lal::diagonal_f64(c, m, rp, ci, v, d);
}
