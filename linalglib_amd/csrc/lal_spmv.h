// Row-block CSR kernels shared by SpMV, residual and the smoothers.
//
// A workgroup of 256 lanes owns a contiguous block of rows [r0, r1) chosen by
// the analysis (at most 256 rows and, unless a single row is longer, at most
// CAP nonzeros).  The block's nonzero range is staged through LDS in chunks of
// CAP entries with coalesced loads: the matrix value and the gathered x value
// of every nonzero land side by side, so the row sums read LDS only.  With
// G = 1 each row is summed by one lane in CSR order, which reproduces the
// host loop bit for bit; sparse blocks (few, long rows) split each row over a
// group of G lanes and combine the partial sums with a fixed butterfly.
#pragma once

#include "lal_columns.h"
#include "lal_internal.h"

#include <vector>

struct lal_csrmv_info
{
    int  m        = 0;
    int  nnz      = 0;
    int  nblocks  = 0;
    int  exact    = 0;       // 1: sequential row sums (bit-identical to the host)
    int  by_nnz   = 0;       // fast path: lanes gather x over consecutive nonzeros
                             // (rectangular transfer operators) instead of per row
    int  win      = 4;       // widest 4-aligned nonzero window of a block (<= 2052)
    int  keep     = 0;       // fast path: the matrix is read with
                             // cache-allocating loads instead of streaming
                             // ones, in FP64 (1) and in FP32 (2)
    int* d_blocks = nullptr; // nblocks + 1 row offsets, then per block
                             // {r0, r1, row_ptr[r0], row_ptr[r1]} at
                             // lal::block_meta_offset(nblocks)
    // 16-bit columns (fast path of the operators a hierarchy owns): entry k of
    // block b stores col_ind[k] - d_cbase[b]; null when not built or a block's
    // columns span more than 65535
    unsigned short* d_c16   = nullptr;
    int*            d_cbase = nullptr;
    // Gathered x through LDS (operators a hierarchy asks it for): every block's
    // distinct columns, ascending, as 16-bit offsets from its smallest one from
    // d_list[lal::list_start()] on (an odd list's last one twice); per nonzero four times its
    // column's place in that list; per block {list length | lal::list_split() << 12 |
    // log2 of the lanes per row << 24, smallest column}.  list_max: the longest
    // list; 0 when not built (a block spans more than 131,072 columns or holds
    // more than 2044 nonzeros).
    unsigned short* d_lpos   = nullptr;
    unsigned short* d_list   = nullptr;
    int*            d_lmeta  = nullptr;
    int             list_max = 0;
    bool            list_far = false; // some offset is 65536 or more
    // room for nb blocks, in the arena or an allocation of its own
    int arrays(lal::arena* mem, int nb);
    bool owned = true; // d_blocks is this descriptor's to free (else, as the
                       // 16-bit columns always, it lies in a hierarchy's arena)
};

namespace lal
{
    // Position (in ints, a multiple of 4) of the per-block quadruples in the
    // descriptor's block array.
    __host__ __device__ inline size_t block_meta_offset(int nblocks)
    {
        return ((size_t)nblocks + 1 + 3) & ~(size_t)3;
    }

    constexpr int SPMV_THREADS = 256;

    // A matrix pattern to analyse: d gets its row blocks and, with want16 and
    // where the blocks allow it, its 16-bit columns; check_n >= 0: every
    // column must lie in [0, check_n).
    struct rb_request
    {
        lal_csrmv_info* d;
        const int*      rp;
        const int*      ci;
        int             m, nnz;
        bool            want16;
        int             check_n;
        bool            want_list = false; // with want16: the blocks' column lists too
    };
    // The same as the analysis kernels see it.
    struct rb_op
    {
        const int*      rp;
        const int*      ci;
        int*            blocks;
        unsigned short* c16;
        int*            cbase;
        unsigned short* lpos;
        unsigned short* list;
        int*            lmeta;
        int             m, nnz, cap;
        int             tile0, ntiles; // its row tiles
        int             blk0, ub;      // its blocks at most, in the columns' grid
    };
    // Analyses every request in one pass over the device (blocks until the
    // results are known).  mem: where the descriptors' arrays lie (null: their
    // own allocations, without 16-bit columns).
    int analyse(lal_context* c, const std::vector<rb_request>& req, arena* mem, arena* tmp);

    // What a hierarchy's operators read with cache-allocating loads may hold
    // (values and column indices at the precision of the call): three quarters
    // of MI355X's 256 MB Infinity Cache, leaving room for the vectors.
    constexpr size_t CACHE_KEEP_BYTES = (size_t)192 << 20;

    template <typename T>
    struct spmv_cap
    {
        static constexpr int value = 2048;
    };

    // log2 of the lanes per row for a block of `rows` rows: the largest power
    // of two up to 64 with which the rows fill at most SPMV_THREADS lanes, one
    // from 128 rows on.
    __device__ __forceinline__ int spmv_group_log(int rows)
    {
        const int up = 32 - __clz(rows - 1); // rows <= 2^up (rows 1: clz(0) is 32)
        return rows >= 128 ? 0 : rows <= 4 ? 6 : 8 - up;
    }

    // Lanes per row; exact: always one.
    __device__ __forceinline__ int spmv_group(int rows, int exact)
    {
        return exact ? 1 : 1 << spmv_group_log(rows);
    }

    // Where a block's column list starts: behind the lists of the blocks
    // before it, which have no more entries than nonzeros, and 8-byte aligned.
    __host__ __device__ inline size_t list_start(int base, int block)
    {
        return (size_t)(base & ~3) + 4 * (size_t)block;
    }

    template <typename T>
    __device__ __forceinline__ T group_sum(T v, int g)
    {
        for(int o = g >> 1; o > 0; o >>= 1)
            v += __shfl_xor(v, o, 64);
        return v;
    }

    __device__ __forceinline__ void block_rows(const int* __restrict__ blocks, int m, int tile,
                                               int* r0, int* r1)
    {
        if(blocks)
        {
            *r0 = blocks[tile];
            *r1 = blocks[tile + 1];
        }
        else
        {
            *r0 = tile * SPMV_THREADS;
            *r1 = min(m, *r0 + SPMV_THREADS);
        }
    }

    inline int spmv_grid(const lal_csrmv_info* d, int m)
    {
        return d ? d->nblocks : (m + SPMV_THREADS - 1) / SPMV_THREADS;
    }
}
