// Sparse products of the SA-AMG setup: transpose (R = P^T) and the two-pass
// hash SpGEMM used for the Galerkin product A_c = R (A P).
//
// Transpose: count, scan, scatter, then each row of the result is sorted by
// column, which gives the stable order of backend/host/host_csr2csc.cpp:30-75.
//
// SpGEMM: rows of C are binned on the device by their product count into LDS
// hash tables of H = 64 ... 4096 slots (open addressing, linear probing,
// slots claimed with atomicCAS); rows beyond that get a table in global
// memory.  A table is built by 8 to 64 lanes (the symbolic pass's large
// key-only ones by a workgroup).  The numeric pass searches the slots of
// several A entries' B rows at once but adds their products in A-row order;
// the columns of one B row are distinct, so every C entry receives at most one
// contribution per A entry and is folded in A-row-then-B-row order from its
// first product -- the exact accumulation of
// backend/host/host_csrgemm.cpp:91-183.  The table is then compacted and each
// entry is placed by its rank, giving ascending columns.
#include "lal_internal.h"

#include <algorithm>
#include <vector>

namespace
{
    // ------------------------------------------------------------ transpose
    // Entries per column, and each entry's place among its column's (in order
    // of arrival; the rows are sorted later): the atomic's return value, so
    // that the scatter needs none of its own.
    // A workgroup counts 2048 entries in an LDS table first (neighbouring rows
    // share most of their columns) and takes its places per distinct column
    // with one global atomic each: 121^3 diffusion's P, 7.4 million entries,
    // 174 us with an atomic per entry, 93 so.
    constexpr int COL_ITEMS = 8;
    constexpr int COL_SLOTS = 4096;

    __global__ void __launch_bounds__(256)
        col_count_kernel(int nnz, const int* __restrict__ ci, int* __restrict__ cnt,
                         int* __restrict__ place)
    {
        __shared__ int s_key[COL_SLOTS], s_n[COL_SLOTS];
        for(int i = threadIdx.x; i < COL_SLOTS; i += 256)
        {
            s_key[i] = -1;
            s_n[i]   = 0;
        }
        __syncthreads();
        const int k0 = blockIdx.x * (256 * COL_ITEMS) + threadIdx.x;
        int       col[COL_ITEMS], slot[COL_ITEMS], at[COL_ITEMS];
#pragma unroll
        for(int u = 0; u < COL_ITEMS; u++)
            col[u] = k0 + 256 * u < nnz ? ci[k0 + 256 * u] : -1;
        // (at most 2048 distinct columns in 4096 slots: every probe ends)
#pragma unroll
        for(int u = 0; u < COL_ITEMS; u++)
            if(col[u] >= 0)
            {
                unsigned h = ((unsigned)col[u] * 2654435761u) >> 20;
                for(;;)
                {
                    const int seen = atomicCAS(&s_key[h], -1, col[u]);
                    if(seen == -1 || seen == col[u])
                        break;
                    h = (h + 1) & (COL_SLOTS - 1);
                }
                slot[u] = (int)h;
                at[u]   = atomicAdd(&s_n[h], 1);
            }
        __syncthreads();
        for(int i = threadIdx.x; i < COL_SLOTS; i += 256)
            if(s_n[i] > 0)
                s_n[i] = atomicAdd(&cnt[s_key[i]], s_n[i]);
        __syncthreads();
#pragma unroll
        for(int u = 0; u < COL_ITEMS; u++)
            if(col[u] >= 0)
                place[k0 + 256 * u] = s_n[slot[u]] + at[u];
    }

    template <typename T>
    __global__ void __launch_bounds__(256)
        transpose_scatter_kernel(int m, const int* __restrict__ rp, const int* __restrict__ ci,
                                 const T* __restrict__ v, const int* __restrict__ trp,
                                 const int* __restrict__ place, int* __restrict__ tci,
                                 T* __restrict__ tv)
    {
        // 4 lanes per row
        const int i = blockIdx.x * 64 + (int)(threadIdx.x >> 2);
        if(i >= m)
            return;
        for(int j = rp[i] + (int)(threadIdx.x & 3); j < rp[i + 1]; j += 4)
        {
            const int pos = trp[ci[j]] + place[j];
            tci[pos]      = i;
            tv[pos]       = v[j];
        }
    }

    // Sorts a row of n <= K G entries by column, stably, with the G lanes from gb
    // on: each lane ranks its entries by counting the row's smaller columns, ties
    // broken by position; the columns pass from lane to lane in registers, and
    // every load of the row completes before the first store, so the row is
    // permuted in place.
    template <int G, int K, typename T>
    __device__ __forceinline__ void rank_row(int s, int n, int gl, int gb, int* __restrict__ ci,
                                             T* __restrict__ v)
    {
        int key[K], rank[K];
        T   val[K];
#pragma unroll
        for(int u = 0; u < K; u++)
        {
            const int j = gl + G * u;
            key[u]      = j < n ? ci[s + j] : INT_MAX;
            val[u]      = j < n ? v[s + j] : (T)0;
            rank[u]     = 0;
        }
#pragma unroll
        for(int w = 0; w < K; w++)
        {
            const int top = min(G, n - G * w); // (none beyond the row)
            for(int t = 0; t < top; t++)
            {
                int kt;
                if constexpr(G == 64)
                    kt = __builtin_amdgcn_readlane(key[w], t);
                else
                    kt = __shfl(key[w], gb + t, 64);
#pragma unroll
                for(int u = 0; u < K; u++)
                    if(G * u < n)
                        rank[u] += kt < key[u] || (kt == key[u] && G * w + t < gl + G * u);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for(int u = 0; u < K; u++)
            if(gl + G * u < n)
            {
                ci[s + rank[u]] = key[u];
                v[s + rank[u]]  = val[u];
            }
    }

    constexpr int WAVE_ROW = 256;  // entries of a row that a wavefront ranks
    constexpr int LONG_RUN = 4096; // keys sorted in LDS at a time

    // Row c of the transpose, n entries from s on, by the whole workgroup: its
    // columns are sorted in LDS runs, which are merged pairwise between tci and
    // tmp (every key finds its place in the other run by binary search); the
    // values then come from the matrix itself, the d-th of several equal columns
    // from the d-th entry of column c in that row.
    template <typename T>
    __device__ void long_row(int c, int s, int n, int* s_key, int* tci, T* tv, int* tmp,
                             const int* __restrict__ rp, const int* __restrict__ ci,
                             const T* __restrict__ v)
    {
        const int tid = (int)threadIdx.x;
        for(int r0 = 0; r0 < n; r0 += LONG_RUN)
        {
            const int len = min(LONG_RUN, n - r0);
            int       pow = 256;
            while(pow < len)
                pow <<= 1;
            for(int t = tid; t < pow; t += 256)
                s_key[t] = t < len ? tci[s + r0 + t] : INT_MAX;
            __syncthreads();
            for(int k = 2; k <= pow; k <<= 1)
                for(int j = k >> 1; j > 0; j >>= 1)
                {
                    for(int t = tid; t < pow / 2; t += 256)
                    {
                        const int at = 2 * t - (t & (j - 1)), x = s_key[at], y = s_key[at + j];
                        if((x > y) == ((at & k) == 0))
                        {
                            s_key[at]     = y;
                            s_key[at + j] = x;
                        }
                    }
                    __syncthreads();
                }
            for(int t = tid; t < len; t += 256)
                tci[s + r0 + t] = s_key[t];
            __syncthreads();
        }
        int *src = tci + s, *dst = tmp + s;
        for(unsigned run = LONG_RUN; run < (unsigned)n; run <<= 1)
        {
            for(unsigned e = tid; e < (unsigned)n; e += 256)
            {
                const int      key  = src[e];
                const unsigned pair = e & ~(2 * run - 1), mid = min(pair + run, (unsigned)n);
                const bool     left = e < mid;
                // the other run's keys that come before this one
                unsigned lo = left ? mid : pair, hi = left ? min(pair + 2 * run, (unsigned)n) : mid;
                const unsigned first = lo;
                while(lo < hi)
                {
                    const unsigned m = (lo + hi) >> 1;
                    if(left ? src[m] < key : src[m] <= key)
                        lo = m + 1;
                    else
                        hi = m;
                }
                dst[(left ? e : pair + (e - mid)) + (lo - first)] = key;
            }
            __syncthreads();
            int* const t = src;
            src          = dst;
            dst          = t;
        }
        if(src != tci + s)
        {
            for(int e = tid; e < n; e += 256)
                tci[s + e] = src[e];
            __syncthreads();
        }
        for(int e = tid; e < n; e += 256)
        {
            const int i = tci[s + e];
            int       d = 0;
            while(d < e && tci[s + e - d - 1] == i)
                d++;
            for(int j = rp[i]; j < rp[i + 1]; j++)
                if(ci[j] == c && d-- == 0)
                {
                    tv[s + e] = v[j];
                    break;
                }
        }
        __syncthreads();
    }

    // Sorts each row of the transpose by column with G lanes per row (16 for rows
    // of up to 32 entries on average, else a wavefront).  Rows of more than K G
    // entries and up to 256 are ranked by the whole wavefront, longer ones sorted
    // by the workgroup, its rows one after the other (tmp: an int per entry; rp,
    // ci, v: the matrix).
    // Bound by the ranking's instructions: rows of 22 entries (121^3 diffusion's
    // R, 341,000 rows) took 236 us with a wavefront each, 125 with 16 lanes.  A
    // transpose with 2000 rows of 200 entries among 98,000 of 8: 202 us (with the
    // insertion sort from 129 entries on 3170, with a wavefront for every row 258).
    // Graph of 60,000 rows, one of 28,000 entries: 3.9 ms, 56 s with one lane's
    // insertion sort (42 s while the entries arrived in another order).
    template <int G, int K, typename T>
    __global__ void __launch_bounds__(256)
        row_sort_kernel(int m, const int* __restrict__ trp, int* tci, T* tv, int* tmp,
                        const int* __restrict__ rp, const int* __restrict__ ci,
                        const T* __restrict__ v)
    {
        __shared__ int s_key[LONG_RUN];
        const int      lane = (int)threadIdx.x & 63, gl = (int)threadIdx.x % G;
        const int      first = blockIdx.x * (256 / G), i = first + (int)threadIdx.x / G;
        const int      s = i < m ? trp[i] : 0, n = i < m ? trp[i + 1] - s : 0;
        if(n > 1 && n <= K * G)
            rank_row<G, K>(s, n, gl, lane - gl, tci, tv);
        if constexpr(K * G < WAVE_ROW)
            for(unsigned long long todo = __ballot(gl == 0 && n > K * G && n <= WAVE_ROW);
                todo != 0; todo &= todo - 1)
            {
                const int t = __ffsll((long long)todo) - 1;
                rank_row<64, WAVE_ROW / 64>(__builtin_amdgcn_readlane(s, t),
                                            __builtin_amdgcn_readlane(n, t), lane, 0, tci, tv);
            }
        if(!__syncthreads_or(n > WAVE_ROW))
            return;
        for(int c = first; c < min(m, first + 256 / G); c++)
        {
            const int at = trp[c], len = trp[c + 1] - at; // (uniform)
            if(len > WAVE_ROW)
                long_row(c, at, len, s_key, tci, tv, tmp, rp, ci, v);
        }
    }

    // -------------------------------------------------------------- SpGEMM
    __global__ void __launch_bounds__(256)
        products_kernel(int m, const int* __restrict__ arp, const int* __restrict__ aci,
                        const int* __restrict__ brp, int* __restrict__ prod)
    {
        int i = blockIdx.x * 256 + threadIdx.x;
        if(i >= m)
            return;
        long long p = 0;
        for(int j = arp[i]; j < arp[i + 1]; j++)
        {
            int c = aci[j];
            p += brp[c + 1] - brp[c];
        }
        prod[i] = (int)min(p, (long long)INT_MAX);
    }

    // products_kernel with G lanes per row, for long rows of A: the lanes
    // sum strided parts of the row, the group adds them up (integers: the
    // same count).
    template <int G>
    __global__ void __launch_bounds__(256)
        products_group_kernel(int m, const int* __restrict__ arp, const int* __restrict__ aci,
                              const int* __restrict__ brp, int* __restrict__ prod)
    {
        const int gl = (int)threadIdx.x % G;
        const int i  = blockIdx.x * (256 / G) + (int)threadIdx.x / G;
        if(i >= m)
            return;
        long long p = 0;
        for(int j = arp[i] + gl; j < arp[i + 1]; j += G)
        {
            int c = aci[j];
            p += brp[c + 1] - brp[c];
        }
#pragma unroll
        for(int o = G / 2; o > 0; o >>= 1)
            p += __shfl_xor(p, o, 64);
        if(gl == 0)
            prod[i] = (int)min(p, (long long)INT_MAX);
    }

    __device__ __forceinline__ int slot_of(int col, int hmask)
    {
        return (int)(((unsigned)col * 0x9E3779B1u) >> 7) & hmask;
    }

    // Orders one step's table updates before the next step's reads across
    // the lanes of the wave: LDS tables need workgroup scope, tables in global
    // memory agent scope (the L1 is not coherent with the atomics in L2).
    template <bool GLOBAL>
    __device__ __forceinline__ void wave_sync_mem()
    {
        if(GLOBAL)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        else
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        if(GLOBAL)
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        else
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }

    // One wavefront builds row `row` of C in a table of H slots (H a power of
    // two, at least 64 and at least twice the row's distinct columns).
    //
    // The numeric pass sizes the table by the row's nonzero count from the
    // symbolic pass.  Should a caller pass a row pointer that undercounts a
    // row, the probing stops after H slots and the row is cut to its length,
    // *err is set, and no slot or output entry outside the row is touched.
    template <bool NUMERIC, bool GLOBAL>
    __device__ void spgemm_row(int row, int* keys, double* vals, int H, int lane,
                               const int* __restrict__ arp, const int* __restrict__ aci,
                               const double* __restrict__ av, const int* __restrict__ brp,
                               const int* __restrict__ bci, const double* __restrict__ bv,
                               const int* __restrict__ crp, int* __restrict__ cout_,
                               double* __restrict__ cval, int* __restrict__ err)
    {
        const int hmask = H - 1;
        for(int s = lane; s < H; s += 64)
            keys[s] = -1;
        wave_sync_mem<GLOBAL>();
        int local = 0;
        for(int j = arp[row]; j < arp[row + 1]; j++)
        {
            const int    ca = aci[j];
            const double va = NUMERIC ? 1.0 * av[j] : 0.0;
            const int    be = brp[ca + 1];
            for(int p = brp[ca] + lane; p < be; p += 64)
            {
                const int col = bci[p];
                int       h   = slot_of(col, hmask);
                for(int probe = 0;; probe++)
                {
                    if(probe == H)
                    {
                        *err = 1; // table full: the row pointer undercounts this row
                        break;
                    }
                    int old = atomicCAS(&keys[h], -1, col);
                    if(old == -1)
                    {
                        local++;
                        if(NUMERIC)
                            vals[h] = va * bv[p];
                        break;
                    }
                    if(old == col)
                    {
                        if(NUMERIC)
                            vals[h] += va * bv[p];
                        break;
                    }
                    h = (h + 1) & hmask;
                }
            }
            wave_sync_mem<GLOBAL>();
        }
        if(!NUMERIC)
        {
            int total = lal::wave_sum(local);
            if(lane == 0)
                cout_[row] = total;
            return;
        }
        // compact the occupied slots into [0, nnz) in place
        int                      base  = 0;
        const unsigned long long below = (1ull << lane) - 1ull;
        for(int s0 = 0; s0 < H; s0 += 64)
        {
            const int          s     = s0 + lane;
            const int          k     = keys[s];
            const double       v     = vals[s];
            const bool         valid = k != -1;
            unsigned long long mask  = __ballot(valid);
            wave_sync_mem<GLOBAL>();
            if(valid)
            {
                int pos   = base + __popcll(mask & below);
                keys[pos] = k;
                vals[pos] = v;
            }
            base += __popcll(mask);
            wave_sync_mem<GLOBAL>();
        }
        const int nnz = base;
        const int out = crp[row];
        const int len = crp[row + 1] - out;
        if(nnz != len && lane == 0)
            *err = 1;
        for(int e = lane; e < nnz; e += 64)
        {
            const int k = keys[e];
            int       r = 0;
            for(int t = 0; t < nnz; t++)
                r += keys[t] < k;
            if(r < len)
            {
                cout_[out + r] = k;
                cval[out + r]  = vals[e];
            }
        }
    }

    // The bins of one launch: nr rows with tables of H slots (a power of two, at
    // least 64) from workgroup `first` on.
    struct group_bins
    {
        struct one
        {
            const int* rows;
            int        nr, H, first;
        };
        one b[10];
        int n = 0, blocks = 0, max_h = 0;
        void add(const int* rows, int nr, int H, int rpb)
        {
            b[n++] = {rows, nr, H, blocks};
            blocks += (nr + rpb - 1) / rpb;
            max_h = std::max(max_h, H);
        }
    };

    // Rows of C in LDS tables: G lanes per row, L of them per B row.
    //
    // Bound by latency: a step (one A entry and its B row) is a chain of
    // dependent loads and LDS round trips, and the coarse levels have few and
    // long rows.  So G lanes load G entries of the A row with their B-row
    // bounds at once, and S * U steps are taken together: S = G / L groups of
    // lanes side by side, U steps per group in flight, first their B-row loads,
    // then their slot searches (which slot a column gets does not depend on
    // the order), and only then, in A-row order, their additions, as LDS adds
    // without a return value.  The LDS executes one wave's instructions in
    // order and the columns of one step are distinct, so every C entry is
    // folded in A-row-then-B-row order; slots start at -0.0, to which adding
    // the first product is exact, so the fold is the one from the first
    // product.  A B row longer than L is several steps.
    //
    // AHEAD: the next batch's B-row loads are issued before this batch's LDS
    // work.  It shortens a row's chain and costs registers and occupancy, so
    // it is for launches of few rows (launch_group).
    template <int G, int L, bool NUMERIC, bool AHEAD>
    __global__ void __launch_bounds__(256)
        spgemm_group_kernel(group_bins bins, const int* __restrict__ arp,
                            const int* __restrict__ aci,
                            const double* __restrict__ av, const int* __restrict__ brp,
                            const int* __restrict__ bci, const double* __restrict__ bv,
                            const int* __restrict__ crp, int* __restrict__ cout_,
                            double* __restrict__ cval, int* __restrict__ err)
    {
        static_assert(G <= 64 && L <= G && (G & (G - 1)) == 0 && (L & (L - 1)) == 0);
        constexpr int S = G / L, U = S >= 4 ? 2 : 4;
        constexpr unsigned long long GMASK = G == 64 ? ~0ull : (1ull << (G % 64)) - 1ull;
        typedef int   int4v __attribute__((ext_vector_type(4)));
        // per row of the workgroup: H values (numeric pass), H keys
        extern __shared__ __attribute__((aligned(16))) unsigned char s_tab[];
        int bin = 0;
        while(bin + 1 < bins.n && bins.b[bin + 1].first <= (int)blockIdx.x)
            bin++;
        const int H     = bins.b[bin].H;
        const int hmask = H - 1;
        const int rpb   = (int)blockDim.x / G;
        const int grp   = (int)threadIdx.x / G;
        const int gl    = (int)threadIdx.x % G;         // lane in the group
        const int gb    = ((int)threadIdx.x & 63) - gl; // the group's first lane
        const int sl    = gl % L, sg = gl / L;          // lane of the step, step of the batch
        const int r     = ((int)blockIdx.x - bins.b[bin].first) * rpb + grp;
        if(r >= bins.b[bin].nr)
            return;
        const int row  = bins.b[bin].rows[r];
        double*   vals = NUMERIC ? reinterpret_cast<double*>(s_tab) + (size_t)grp * H : nullptr;
        int*      keys = reinterpret_cast<int*>(s_tab + (NUMERIC ? sizeof(double) * rpb * H : 0)) +
                    (size_t)grp * H;
        for(int s = gl; s < H / 4; s += G)
            reinterpret_cast<int4v*>(keys)[s] = int4v{-1, -1, -1, -1};
        if(NUMERIC)
            for(int s = gl; s < H; s += G)
                vals[s] = -0.0;
        wave_sync_mem<false>();
        // lane t's value of v, for the whole group (a wavefront taking its
        // steps one by one reads the lane as a scalar)
        auto lane_value = [&](auto v, int t) {
            if constexpr(S == 1 && G == 64)
                return lal::wave_lane(v, __builtin_amdgcn_readfirstlane(t));
            else
                return __shfl(v, gb + t, 64);
        };
        int       local = 0;
        const int rs = arp[row], re = arp[row + 1];
        for(int j0 = rs; j0 < re; j0 += G)
        {
            const int j  = j0 + gl;
            int       bs = 0, be = 0;
            double    va = 0.0;
            if(j < re)
            {
                const int ca = aci[j];
                if(NUMERIC)
                    va = 1.0 * av[j];
                bs = brp[ca];
                be = brp[ca + 1];
            }
            // steps of this chunk: one per A entry, or more where a B row is
            // longer than L (then `upto` counts the steps through each entry)
            const bool wide  = ((__ballot(be - bs > L) >> gb) & GMASK) != 0;
            int        steps = min(G, re - j0);
            int        upto  = 0;
            if(wide)
            {
                upto = (be - bs + L - 1) / L;
#pragma unroll
                for(int o = 1; o < G; o <<= 1)
                {
                    const int t = __shfl(upto, gb + max(gl - o, 0), 64);
                    upto += gl >= o ? t : 0;
                }
                steps = __shfl(upto, gb + G - 1, 64);
            }
            // entries of the steps s0 .. s0 + S U - 1: columns (-1: none), the
            // B values and the A value of their step
            auto fetch = [&](int s0, int (&col)[U], double (&bval)[U], double (&aval)[U]) {
#pragma unroll
                for(int u = 0; u < U; u++)
                {
                    const int s = s0 + u * S + sg;
                    int       t = min(s, G - 1), off = 0; // A entry, chunk of its B row
                    if(wide)
                    {
                        // t: the entries that end at or before step s
                        if(G == 64 && S == 1)
                            t = min(__popcll(__ballot(upto <= s)), G - 1);
                        else
                        {
                            t = 0;
#pragma unroll
                            for(int o = G / 2; o > 0; o >>= 1)
                            {
                                const int v = __shfl(upto, gb + t + o - 1, 64);
                                t += v <= s ? o : 0;
                            }
                        }
                        const int before = lane_value(upto, max(t - 1, 0));
                        off              = (s - (t > 0 ? before : 0)) * L;
                    }
                    const int  p  = lane_value(bs, t) + off + sl;
                    const int  pe = lane_value(be, t); // every lane takes part
                    const bool ok = s < steps && p < pe;
                    aval[u]       = NUMERIC ? lane_value(va, t) : 0.0;
                    col[u]        = ok ? bci[p] : -1;
                    bval[u]       = NUMERIC && ok ? bv[p] : 0.0;
                }
            };
            int    ncol[U];
            double nbv[U], nav[U];
            if(AHEAD)
                fetch(0, ncol, nbv, nav);
            for(int s0 = 0; s0 < steps; s0 += S * U)
            {
                int      col[U], h[U];
                double   prod[U];
                unsigned pend = 0;
                if(!AHEAD)
                    fetch(s0, ncol, nbv, nav);
#pragma unroll
                for(int u = 0; u < U; u++)
                {
                    prod[u] = nav[u] * nbv[u];
                    col[u]  = ncol[u];
                    h[u]    = slot_of(col[u], hmask);
                    pend |= col[u] >= 0 ? 1u << u : 0u;
                }
                if(AHEAD && s0 + S * U < steps)
                    fetch(s0 + S * U, ncol, nbv, nav);
                const unsigned all = pend;
                for(int probe = 0; pend != 0; probe++)
                {
                    if(probe == H)
                    {
                        *err = 1; // table full: the row pointer undercounts this row
                        break;
                    }
                    int old[U];
#pragma unroll
                    for(int u = 0; u < U; u++)
                        if(pend >> u & 1)
                            old[u] = atomicCAS(&keys[h[u]], -1, col[u]);
#pragma unroll
                    for(int u = 0; u < U; u++)
                        if(pend >> u & 1)
                        {
                            if(old[u] == -1)
                                local++;
                            if(old[u] == -1 || old[u] == col[u])
                                pend &= ~(1u << u);
                            else
                                h[u] = (h[u] + 1) & hmask;
                        }
                }
                if(NUMERIC)
                {
                    const unsigned got = all & ~pend;
#pragma unroll
                    for(int u = 0; u < U; u++)
#pragma unroll
                        for(int k = 0; k < S; k++)
                        {
                            if(sg == k && (got >> u & 1))
                                (void)__hip_atomic_fetch_add(&vals[h[u]], prod[u],
                                                             __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_WORKGROUP);
                            __builtin_amdgcn_wave_barrier();
                        }
                }
            }
        }
        if(!NUMERIC)
        {
#pragma unroll
            for(int o = G / 2; o > 0; o >>= 1)
                local += __shfl_xor(local, o, 64);
            if(gl == 0)
                cout_[row] = local;
            return;
        }
        wave_sync_mem<false>();
        // compact the occupied slots into [0, nnz) in place, eight per lane at
        // a time (an entry never moves up, so the slots a later pass reads
        // are still untouched)
        int                      base  = 0;
        const unsigned long long below = (1ull << gl) - 1ull;
        for(int s0 = 0; s0 < H; s0 += 8 * G)
        {
            int    k[8];
            double v[8];
#pragma unroll
            for(int u = 0; u < 8; u++)
            {
                const int t = s0 + u * G + gl;
                k[u]        = t < H ? keys[t] : -1;
                v[u]        = t < H ? vals[t] : 0.0;
            }
            wave_sync_mem<false>();
#pragma unroll
            for(int u = 0; u < 8; u++)
            {
                const unsigned long long mask = (__ballot(k[u] != -1) >> gb) & GMASK;
                if(k[u] != -1)
                {
                    const int pos = base + __popcll(mask & below);
                    keys[pos]     = k[u];
                    vals[pos]     = v[u];
                }
                base += __popcll(mask);
            }
            wave_sync_mem<false>();
        }
        const int nnz  = base;
        const int nnz4 = (nnz + 3) & ~3; // at most H, a multiple of 4
        if(nnz + gl < nnz4)
            keys[nnz + gl] = INT_MAX;
        wave_sync_mem<false>();
        const int out = crp[row];
        const int len = crp[row + 1] - out;
        if(nnz != len && gl == 0)
            *err = 1;
        // an entry's place is the number of smaller columns, four per read
        for(int e = gl; e < nnz; e += G)
        {
            const int    k  = keys[e];
            int          rk = 0;
            const int4v* k4 = reinterpret_cast<const int4v*>(keys);
            for(int t = 0; t < nnz4 / 4; t++)
            {
                const int4v q = k4[t];
                rk += (q.x < k) + (q.y < k) + (q.z < k) + (q.w < k);
            }
            if(rk < len)
            {
                cout_[out + rk] = k;
                cval[out + rk]  = vals[e];
            }
        }
    }

    // Distinct columns of one row of C per workgroup, in a key table of H
    // slots: the symbolic pass's rows of more than 512 products or so.  The
    // count does not depend on the order, so 32 groups of 8 lanes take the A
    // row's entries side by side, four B-row entries per lane in flight; a
    // wavefront walking such a row alone was a chain of some hundred
    // dependent steps on a tenth of the chip.
    template <int H>
    __global__ void __launch_bounds__(256)
        spgemm_count_kernel(const int* __restrict__ rows, const int* __restrict__ arp,
                            const int* __restrict__ aci, const int* __restrict__ brp,
                            const int* __restrict__ bci, int* __restrict__ cout_,
                            int* __restrict__ err)
    {
        constexpr int G = 8, U = 4, hmask = H - 1;
        __shared__ int s_keys[H];
        __shared__ int s_sum[4];
        const int tid = (int)threadIdx.x, gl = tid % G;
        const int row = rows[blockIdx.x];
        const int re  = arp[row + 1];
        int       j   = arp[row] + tid / G;
        for(int s = tid; s < H; s += 256)
            s_keys[s] = -1;
        __syncthreads();
        int local = 0;
        for(; j < re; j += 256 / G)
        {
            const int ca = aci[j];
            const int be = brp[ca + 1];
            for(int p0 = brp[ca] + gl; p0 < be; p0 += U * G)
            {
                int      col[U], h[U];
                unsigned pend = 0;
#pragma unroll
                for(int u = 0; u < U; u++)
                {
                    const int p = p0 + u * G;
                    col[u]      = p < be ? bci[p] : -1;
                }
#pragma unroll
                for(int u = 0; u < U; u++)
                {
                    h[u] = slot_of(col[u], hmask);
                    pend |= col[u] >= 0 ? 1u << u : 0u;
                }
                for(int probe = 0; pend != 0; probe++)
                {
                    if(probe == H)
                    {
                        *err = 1;
                        break;
                    }
                    int old[U];
#pragma unroll
                    for(int u = 0; u < U; u++)
                        if(pend >> u & 1)
                            old[u] = atomicCAS(&s_keys[h[u]], -1, col[u]);
#pragma unroll
                    for(int u = 0; u < U; u++)
                        if(pend >> u & 1)
                        {
                            if(old[u] == -1)
                                local++;
                            if(old[u] == -1 || old[u] == col[u])
                                pend &= ~(1u << u);
                            else
                                h[u] = (h[u] + 1) & hmask;
                        }
                }
            }
        }
        local = lal::wave_sum(local);
        if((tid & 63) == 0)
            s_sum[tid >> 6] = local;
        __syncthreads();
        if(tid == 0)
            cout_[row] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
    }

    template <bool NUMERIC>
    __global__ void __launch_bounds__(64)
        spgemm_global_kernel(int nrows, const int* __restrict__ rows,
                             const long long* __restrict__ toff, int* __restrict__ tkeys,
                             double* __restrict__ tvals, const int* __restrict__ arp,
                             const int* __restrict__ aci, const double* __restrict__ av,
                             const int* __restrict__ brp, const int* __restrict__ bci,
                             const double* __restrict__ bv, const int* __restrict__ crp,
                             int* __restrict__ cout_, double* __restrict__ cval,
                             int* __restrict__ err)
    {
        const int r = blockIdx.x;
        if(r >= nrows)
            return;
        const long long o = toff[r];
        const int       H = (int)(toff[r + 1] - o);
        spgemm_row<NUMERIC, true>(rows[r], tkeys + o, NUMERIC ? tvals + o : nullptr, H,
                            threadIdx.x & 63, arp, aci, av, brp, bci, bv, crp, cout_, cval, err);
    }

    // LDS tables: up to 4096 slots with values (numeric pass, 48 KB), up to
    // 32768 keys alone (symbolic pass, 128 KB of the 160 KB of LDS).
    constexpr int kLdsMaxH    = 4096;
    constexpr int kLdsMaxHSym = 32768;

    // Slots of a row's table: the smallest power of two >= 64 holding twice
    // the row's bound on distinct columns (its product or nonzero count,
    // capped by the column count of C).
    __device__ __forceinline__ long long table_slots(int prod, int ncols)
    {
        const long long cap  = ncols > 1 ? ncols : 1;
        const long long need = 2LL * (prod < cap ? prod : cap);
        return need <= 64 ? 64 : 1LL << (64 - __clzll(need - 1));
    }

    // Rows of C grouped by hash-table size.
    struct spgemm_plan
    {
        std::vector<int>  bin_start; // per LDS bin (H = 64 << b), into d_rows
        int               n_lds    = 0;
        int               n_global = 0;
        int               g        = 8; // lanes per A row and per B row
        int               l        = 8; // (launch_group)
        std::vector<long long> toff; // global table offsets (n_global + 1)
        int*              d_prod   = nullptr; // products per row (symbolic plan)
        int*              d_part   = nullptr; // row offsets per bin and workgroup
        int*              d_rows   = nullptr; // LDS-bin rows, then global rows
        long long*        d_gsl    = nullptr; // table sizes of the global rows
        long long*        d_toff   = nullptr;
        int*              d_keys   = nullptr;
        double*           d_vals   = nullptr;
    };

    constexpr int kBins = 10; // 64 .. 32768 (above 4096 only for the symbolic pass)

    // Bin of row i of C, or -1 for a row the pass skips: bins 0 .. kBins-1
    // hold LDS tables of 64 << b slots, bin kBins tables in global memory
    // (*slots gets the row's table size).  The symbolic pass sizes a row by
    // its product count (`prod`) and skips rows without products; the
    // numeric pass sizes every row by its nonzero count from the symbolic
    // pass (`crp`), empty rows included, so that a row pointer which
    // undercounts them is detected.
    __device__ __forceinline__ int size_bin(int p, bool skip_empty, int ncols, int max_h,
                                            long long* slots)
    {
        if(skip_empty && p <= 0)
            return -1;
        const long long H = table_slots(p > 0 ? p : 0, ncols);
        *slots            = H;
        // (H is a power of two of 64 or more)
        return H > max_h ? kBins : __ffsll(H) - 7;
    }
    __device__ __forceinline__ int row_bin(int i, const int* __restrict__ prod,
                                           const int* __restrict__ crp, int ncols, int max_h,
                                           long long* slots)
    {
        return size_bin(crp ? crp[i + 1] - crp[i] : prod[i], !crp, ncols, max_h, slots);
    }

    // Rows of a workgroup of the binning kernels (each takes one contiguous
    // range; at most BIN_GROUPS of them, so that one workgroup adds them up).
    constexpr int BIN_GROUPS = 1024;
    inline int bin_rows(int m)
    {
        return std::max(256, ((m + BIN_GROUPS - 1) / BIN_GROUPS + 255) / 256 * 256);
    }

    // part[bin * groups + workgroup] = the workgroup's rows in the bin.  The
    // symbolic pass also clears its counts (rows without products keep the 0).
    __global__ void __launch_bounds__(256)
        bin_count_kernel(int m, int per, const int* __restrict__ prod,
                         const int* __restrict__ crp, int ncols, int max_h,
                         int* __restrict__ part, int* __restrict__ clear)
    {
        __shared__ int s_n[kBins + 1];
        if(threadIdx.x <= kBins)
            s_n[threadIdx.x] = 0;
        __syncthreads();
        const int r0 = blockIdx.x * per, r1 = min(m, r0 + per);
        for(int i = r0 + (int)threadIdx.x; i < r1; i += 256)
        {
            long long H = 0;
            const int b = row_bin(i, prod, crp, ncols, max_h, &H);
            if(b >= 0)
                atomicAdd(&s_n[b], 1);
            if(clear)
                clear[i] = 0;
        }
        if(clear && r1 == m && threadIdx.x == 0)
            clear[m] = 0;
        __syncthreads();
        if(threadIdx.x <= kBins)
            part[threadIdx.x * gridDim.x + blockIdx.x] = s_n[threadIdx.x];
    }

    // One workgroup: the counts, bin after bin, become row offsets (one scan
    // over all of them).  The host's note: the rows of every bin, then *tail
    // (when given).
    __global__ void __launch_bounds__(1024)
        bin_scan_kernel(int groups, int* __restrict__ part, const int* __restrict__ tail,
                        int* note, unsigned seq)
    {
        __shared__ int s_w[16];
        __shared__ int s_first[kBins + 2]; // offset of each bin's first row
        const int      lane = (int)threadIdx.x & 63, wid = (int)threadIdx.x >> 6;
        const int      n     = (kBins + 1) * groups;
        int            carry = 0;
        for(int i0 = 0; i0 < n; i0 += 1024)
        {
            const int i   = i0 + (int)threadIdx.x;
            const int v   = i < n ? part[i] : 0;
            int       inc = v;
#pragma unroll
            for(int o = 1; o < 64; o <<= 1)
            {
                const int q = __shfl_up(inc, o, 64);
                inc += lane >= o ? q : 0;
            }
            if(lane == 63)
                s_w[wid] = inc;
            __syncthreads();
            int off = carry, tot = 0;
            for(int w = 0; w < 16; w++)
            {
                off += w < wid ? s_w[w] : 0;
                tot += s_w[w];
            }
            if(i < n)
            {
                part[i] = off + inc - v;
                if(i % groups == 0)
                    s_first[i / groups] = off + inc - v;
            }
            carry += tot;
            __syncthreads();
        }
        if(threadIdx.x == 0)
            s_first[kBins + 1] = carry;
        __syncthreads();
        if(wid == 0)
            lal::put_note(note, kBins + 2,
                          lane <= kBins                ? s_first[lane + 1] - s_first[lane]
                          : lane == kBins + 1 && tail ? *tail
                                                      : 0,
                          seq);
    }

    // Rows into their bins, at the workgroup's offsets (each row of C is
    // computed on its own, so the order within a workgroup changes no
    // result).  A row of the global bin, whose first position is g0, also
    // records its table size in gslots.
    __global__ void __launch_bounds__(256)
        bin_scatter_kernel(int m, int per, const int* __restrict__ prod,
                           const int* __restrict__ crp, int ncols, int max_h,
                           const int* __restrict__ part, int* __restrict__ rows, int g0,
                           long long* __restrict__ gslots)
    {
        __shared__ int s_at[kBins + 1];
        if(threadIdx.x <= kBins)
            s_at[threadIdx.x] = part[threadIdx.x * gridDim.x + blockIdx.x];
        __syncthreads();
        const int r0 = blockIdx.x * per, r1 = min(m, r0 + per);
        for(int i = r0 + (int)threadIdx.x; i < r1; i += 256)
        {
            long long H = 0;
            const int b = row_bin(i, prod, crp, ncols, max_h, &H);
            if(b < 0)
                continue;
            const int pos = atomicAdd(&s_at[b], 1);
            rows[pos]     = i;
            if(b == kBins)
                gslots[pos - g0] = H;
        }
    }

    // The whole plan of up to PLAN_SMALL rows in one workgroup: a small
    // product's time is its launches (a 25^3 hierarchy build: 318 launches in
    // 2.5 ms).  Row sizes from prod (crp null), from the row pointer crp, or,
    // with SCAN, from the counts in crp, which become the row pointer (m + 1
    // entries).  rows gets the rows bin by bin, gslots the table sizes of those
    // in the last bin, the note what bin_scan_kernel's gets.
    constexpr int PLAN_CHUNKS = 16;
    constexpr int PLAN_SMALL  = PLAN_CHUNKS * 1024 - 1;

    template <bool SCAN>
    __global__ void __launch_bounds__(1024)
        plan_small_kernel(int m, const int* __restrict__ prod, int* __restrict__ crp, int ncols,
                          int max_h, int* __restrict__ rows, long long* __restrict__ gslots,
                          int* __restrict__ clear, int* note, unsigned seq)
    {
        __shared__ int s_w[2][16];
        __shared__ int s_n[kBins + 1], s_at[kBins + 1];
        const int      tid = (int)threadIdx.x, lane = tid & 63, wid = tid >> 6;
        if(tid <= kBins)
            s_n[tid] = 0;
        // (chunks past the last row are skipped by the whole workgroup)
        int p[PLAN_CHUNKS];
#pragma unroll
        for(int k = 0; k < PLAN_CHUNKS; k++)
            if(k * 1024 <= m)
            {
                const int i = k * 1024 + tid;
                p[k]        = i >= m ? 0 : SCAN ? crp[i] : crp ? crp[i + 1] - crp[i] : prod[i];
                if(clear && i <= m)
                    clear[i] = 0;
            }
        __syncthreads();
        int total = 0;
#pragma unroll
        for(int k = 0; k < PLAN_CHUNKS; k++)
            if(k * 1024 <= m)
            {
                const int i = k * 1024 + tid;
                if(SCAN)
                {
                    int inc = p[k];
#pragma unroll
                    for(int o = 1; o < 64; o <<= 1)
                    {
                        const int q = __shfl_up(inc, o, 64);
                        inc += lane >= o ? q : 0;
                    }
                    if(lane == 63)
                        s_w[k & 1][wid] = inc;
                    __syncthreads();
                    int at = total + inc - p[k];
                    for(int w = 0; w < 16; w++)
                    {
                        at += w < wid ? s_w[k & 1][w] : 0;
                        total += s_w[k & 1][w];
                    }
                    if(i <= m)
                        crp[i] = at;
                }
                long long H = 0;
                const int b = i < m ? size_bin(p[k], !SCAN && !crp, ncols, max_h, &H) : -1;
                if(b >= 0)
                    atomicAdd(&s_n[b], 1);
            }
        __syncthreads();
        if(tid <= kBins)
        {
            int at = 0;
            for(int b = 0; b < tid; b++)
                at += s_n[b];
            s_at[tid] = at;
        }
        __syncthreads();
        const int g0 = s_at[kBins];
        __syncthreads();
#pragma unroll
        for(int k = 0; k < PLAN_CHUNKS; k++)
            if(k * 1024 < m)
            {
                long long H = 0;
                const int i = k * 1024 + tid;
                const int b = i < m ? size_bin(p[k], !SCAN && !crp, ncols, max_h, &H) : -1;
                if(b < 0)
                    continue;
                const int pos = atomicAdd(&s_at[b], 1);
                rows[pos]     = i;
                if(b == kBins)
                    gslots[pos - g0] = H;
            }
        if(wid == 0)
            lal::put_note(note, kBins + 2,
                          lane <= kBins ? s_n[lane] : lane == kBins + 1 ? total : 0, seq);
    }

    // Rows of C binned by table size on the device; the host gets the eleven
    // counts and, with `scan` (crp holds the rows' counts and becomes the row
    // pointer), the number of C's entries.  Up to PLAN_SMALL rows are in their
    // lists after one launch, larger products' go there in plan_rows.
    int plan_count(lal_context* c, int m, int n, int* crp, bool numeric, spgemm_plan& P,
                   lal::temps& tmp, int* clear, bool scan, int* total_out, lal::arena* a)
    {
        constexpr int nb = kBins + 1;
        P.bin_start.assign(nb, 0);
        P.n_lds = P.n_global = 0;
        if(m <= 0)
            return LAL_OK;
        const int max_h = numeric ? kLdsMaxH : kLdsMaxHSym;
        unsigned  seq   = 0;
        if(m <= PLAN_SMALL)
        {
            LAL_TRY(tmp.get(&P.d_rows, m));
            LAL_TRY(tmp.get(&P.d_gsl, m));
            seq      = ++c->note_seq;
            auto* fn = scan ? plan_small_kernel<true> : plan_small_kernel<false>;
            fn<<<1, 1024, 0, c->stream>>>(m, P.d_prod, numeric ? crp : nullptr, n, max_h, P.d_rows,
                                          P.d_gsl, clear, c->d_note, seq);
        }
        else
        {
            if(scan)
                LAL_TRY(lal::scan_i32_dev(c, m + 1, crp, a));
            const int per    = bin_rows(m);
            const int groups = (m + per - 1) / per;
            LAL_TRY(tmp.get(&P.d_part, (size_t)nb * groups));
            bin_count_kernel<<<groups, 256, 0, c->stream>>>(
                m, per, P.d_prod, numeric ? crp : nullptr, n, max_h, P.d_part, clear);
            LAL_LAUNCHED();
            seq = ++c->note_seq;
            bin_scan_kernel<<<1, 1024, 0, c->stream>>>(groups, P.d_part, scan ? crp + m : nullptr,
                                                       c->d_note, seq);
        }
        LAL_LAUNCHED();
        int got[nb + 1];
        LAL_TRY(lal::take_note(c, seq, nb + 1, got));
        int total = 0;
        for(int b = 0; b < nb; b++)
        {
            P.bin_start[b] = total;
            total += got[b];
        }
        P.n_lds    = P.bin_start[kBins];
        P.n_global = got[kBins];
        if(total_out)
            *total_out = got[kBins + 1];
        return LAL_OK;
    }

    // The rows' lists where they are not there yet, and the tables of those
    // that need global memory.
    int plan_rows(lal_context* c, int m, int n, const int* crp, bool numeric, spgemm_plan& P,
                  lal::temps& tmp)
    {
        const int total = P.n_lds + P.n_global;
        if(total == 0)
            return LAL_OK;
        if(m > PLAN_SMALL)
        {
            const int per    = bin_rows(m);
            const int groups = (m + per - 1) / per;
            LAL_TRY(tmp.get(&P.d_rows, total));
            if(P.n_global)
                LAL_TRY(tmp.get(&P.d_gsl, P.n_global));
            bin_scatter_kernel<<<groups, 256, 0, c->stream>>>(
                m, per, P.d_prod, numeric ? crp : nullptr, n, numeric ? kLdsMaxH : kLdsMaxHSym,
                P.d_part, P.d_rows, P.n_lds, P.d_gsl);
            LAL_LAUNCHED();
        }
        if(P.n_global)
        {
            P.toff.assign(P.n_global + 1, 0);
            LAL_HIP(hipMemcpyAsync(P.toff.data() + 1, P.d_gsl, sizeof(long long) * P.n_global,
                                   hipMemcpyDeviceToHost, c->stream));
            LAL_HIP(hipStreamSynchronize(c->stream));
            for(int r = 0; r < P.n_global; r++)
                P.toff[r + 1] += P.toff[r];
            const long long slots = P.toff[P.n_global];
            LAL_TRY(tmp.get(&P.d_toff, P.toff.size()));
            LAL_HIP(hipMemcpyAsync(P.d_toff, P.toff.data(), sizeof(long long) * P.toff.size(),
                                   hipMemcpyHostToDevice, c->stream));
            LAL_TRY(tmp.get(&P.d_keys, slots));
            if(numeric)
                LAL_TRY(tmp.get(&P.d_vals, slots));
            // P.toff must outlive the copy to the device
            LAL_HIP(hipStreamSynchronize(c->stream));
        }
        return LAL_OK;
    }

    // Products of every row of C, for the symbolic plan (rows of A averaging
    // 16 or more entries: 16 lanes per row).
    int count_products(lal_context* c, int m, const int* arp, const int* aci, const int* brp,
                       long nnz_a, spgemm_plan& P, lal::temps& tmp)
    {
        if(m <= 0)
            return LAL_OK;
        LAL_TRY(tmp.get(&P.d_prod, m));
        if(nnz_a >= 16L * m)
            products_group_kernel<16><<<(int)(((long)m * 16 + 255) / 256), 256, 0, c->stream>>>(
                m, arp, aci, brp, P.d_prod);
        else
            products_kernel<<<lal::grid_for(m, 256), 256, 0, c->stream>>>(m, arp, aci, brp,
                                                                          P.d_prod);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    // Smallest power of two of 8 .. 64 that holds n entries.
    inline int lanes_for(long n)
    {
        int g = 8;
        while(g < 64 && g < n)
            g <<= 1;
        return g;
    }

    // Rows of C in their tables: l lanes take a B row (its mean length), g lanes
    // the A row (its mean length).  Below 262,144 such lanes (half of
    // what the chip holds) the rows' own chains are the time: they take a
    // wavefront each and load a batch ahead.  121^3 diffusion, numeric pass:
    // level 3's R (A P), 4,400 rows, takes 502 us with the batch ahead and 648
    // without (960 with one step at a time); level 0's, 300,000 rows, 606 with
    // and 484 without (790 with one step at a time).
    inline bool few_rows(int nr, int g)
    {
        return (long)nr * g < 256L * 1024;
    }
    inline size_t table_bytes(int H, bool numeric)
    {
        return (size_t)H * (numeric ? 12 : 4);
    }

    // (one bin, or several of few rows)
    template <bool NUMERIC>
    void launch_group(lal_context* c, const int* const* rows, const int* nr, const int* H, int n,
                      int g, int l, const int* arp, const int* aci, const double* av,
                      const int* brp, const int* bci, const double* bv, const int* crp,
                      int* cout_, double* cval)
    {
        const bool few = n > 1 || few_rows(nr[0], g);
        if(few)
            g = 64;
        g = std::max(g, l);
        // The counting pass, whose order does not matter: twice the lanes where the
        // tables of 256 would not let eight workgroups share a CU's LDS.  kNN
        // graphs, 12 neighbours (512 and 1024 slots, 16 lanes by the mean), kernel
        // time: 60,000 points 56 -> 42 us, 150,001 184 -> 127, 300,000 334 -> 233
        // (four times the lanes 45, 134, 251).  7-point operators (128 slots, 8
        // lanes, 16 KB) stay: 100^3 91 us, 199 with four times.
        if(!NUMERIC && !few && g < 64 && table_bytes(H[0], false) * (256 / g) > 20 * 1024)
            g <<= 1;
        // up to 256 lanes and 48 KB of tables per workgroup; a row for each
        // where several bins share the launch.  Rows much longer than the mean
        // that chose g (a matrix of few long rows among many short ones) get as
        // many lanes as leave room for their tables.
        int        nt  = n > 1 ? 64 : 256;
        const auto big = [&] { return table_bytes(H[0], NUMERIC) * (nt / g) > 48 * 1024; };
        while(nt > 64 && big())
            nt >>= 1;
        while(g < nt && big())
            g <<= 1;
        const int  rpb = nt / g;
        group_bins bins;
        for(int k = 0; k < n; k++)
            bins.add(rows[k], nr[k], H[k], rpb);
        const size_t lds = table_bytes(bins.max_h, NUMERIC) * rpb;
        const int    nb  = bins.blocks;
#define LAL_SPGEMM_GROUP(GG, LL, AHEAD)                                                      \
    case (AHEAD ? 65536 : 0) + GG * 128 + LL:                                                \
        spgemm_group_kernel<GG, LL, NUMERIC, AHEAD><<<nb, nt, lds, c->stream>>>(             \
            bins, arp, aci, av, brp, bci, bv, crp, cout_, cval, c->d_flag);                  \
        break;
        switch((few ? 65536 : 0) + g * 128 + l)
        {
            LAL_SPGEMM_GROUP(8, 8, false)
            LAL_SPGEMM_GROUP(16, 8, false)
            LAL_SPGEMM_GROUP(16, 16, false)
            LAL_SPGEMM_GROUP(32, 8, false)
            LAL_SPGEMM_GROUP(32, 16, false)
            LAL_SPGEMM_GROUP(32, 32, false)
            LAL_SPGEMM_GROUP(64, 8, false)
            LAL_SPGEMM_GROUP(64, 16, false)
            LAL_SPGEMM_GROUP(64, 32, false)
            LAL_SPGEMM_GROUP(64, 64, false)
            LAL_SPGEMM_GROUP(64, 8, true)
            LAL_SPGEMM_GROUP(64, 16, true)
            LAL_SPGEMM_GROUP(64, 32, true)
            LAL_SPGEMM_GROUP(64, 64, true)
        }
#undef LAL_SPGEMM_GROUP
    }

    template <bool NUMERIC>
    int run_plan(lal_context* c, const spgemm_plan& P, const int* arp, const int* aci,
                 const double* av, const int* brp, const int* bci, const double* bv,
                 const int* crp, int* cout_, double* cval)
    {
        // Bins of few rows share a launch, longest rows first: one after the
        // other, each is as long as its longest row and leaves most of the chip
        // idle (level 4 of a 121^3 diffusion hierarchy, 464 rows in four bins:
        // 450 us apart, 175 together).  Every workgroup then has room for the
        // largest table, so a launch takes rows up to four times what the chip
        // holds at once (once: 10.65 ms for the whole build, four times: 10.51).
        const int* rows[kBins];
        int        nrs[kBins], hs[kBins], n = 0;
        long       joined = 0;
        const auto flush  = [&]() -> int {
            if(n == 0)
                return LAL_OK;
            launch_group<NUMERIC>(c, rows, nrs, hs, n, P.g, P.l, arp, aci, av, brp, bci, bv, crp,
                                  cout_, cval);
            n      = 0;
            joined = 0;
            LAL_LAUNCHED();
            return LAL_OK;
        };
        for(int b = kBins - 1; b >= 0; b--)
        {
            const int n0 = P.bin_start[b], nr = P.bin_start[b + 1] - n0, H = 64 << b;
            if(nr == 0)
                continue;
#define LAL_SPGEMM_COUNT(HH)                                                                 \
    spgemm_count_kernel<HH><<<nr, 256, 0, c->stream>>>(P.d_rows + n0, arp, aci, brp, bci,     \
                                                       cout_, c->d_flag)
            // the symbolic pass's tables of 2048 slots and more (alone beyond
            // 4096), and smaller ones of so few rows that the chip holds a
            // workgroup for each: a workgroup per row
            if(!NUMERIC && (H >= 2048 || (H >= 512 && nr <= 2048)))
            {
                switch(b)
                {
                case 3: LAL_SPGEMM_COUNT(512); break;
                case 4: LAL_SPGEMM_COUNT(1024); break;
                case 5: LAL_SPGEMM_COUNT(2048); break;
                case 6: LAL_SPGEMM_COUNT(4096); break;
                case 7: LAL_SPGEMM_COUNT(8192); break;
                case 8: LAL_SPGEMM_COUNT(16384); break;
                default: LAL_SPGEMM_COUNT(32768); break;
                }
                LAL_LAUNCHED();
                continue;
            }
#undef LAL_SPGEMM_COUNT
            const int  largest = n > 0 ? hs[0] : H;
            const long held =
                4L * c->num_cu * (long)(160 * 1024 / table_bytes(largest, NUMERIC));
            if(n > 0 && (!few_rows(nr, P.g) || joined + nr > held))
                LAL_TRY(flush());
            rows[n] = P.d_rows + n0;
            nrs[n]  = nr;
            hs[n]   = H;
            n++;
            joined += nr;
            if(!few_rows(nr, P.g))
                LAL_TRY(flush());
        }
        LAL_TRY(flush());
        if(P.n_global)
        {
            spgemm_global_kernel<NUMERIC><<<P.n_global, 64, 0, c->stream>>>(
                P.n_global, P.d_rows + P.n_lds, P.d_toff, P.d_keys, P.d_vals, arp, aci, av, brp,
                bci, bv, crp, cout_, cval, c->d_flag);
            LAL_LAUNCHED();
        }
        return LAL_OK;
    }
}

namespace lal
{
    template <typename T>
    int transpose_t(lal_context* c, int m, int n, int nnz, const int* rp, const int* ci,
                    const T* v, int* trp, int* tci, T* tv, arena* a)
    {
        temps tmp(c, a);
        LAL_HIP(hipMemsetAsync(trp, 0, sizeof(int) * (n + 1), c->stream));
        int* place = nullptr;
        if(nnz > 0)
        {
            LAL_TRY(tmp.get(&place, nnz));
            col_count_kernel<<<grid_for(nnz, 256 * COL_ITEMS), 256, 0, c->stream>>>(nnz, ci, trp,
                                                                                    place);
            LAL_LAUNCHED();
        }
        LAL_TRY(scan_i32_dev(c, n + 1, trp, a));
        if(nnz == 0)
            return LAL_OK;
        transpose_scatter_kernel<T><<<grid_for(m, 64), 256, 0, c->stream>>>(m, rp, ci, v, trp,
                                                                            place, tci, tv);
        LAL_LAUNCHED();
        if(nnz <= 32L * n)
            row_sort_kernel<16, 8, T><<<(n + 15) / 16, 256, 0, c->stream>>>(n, trp, tci, tv, place, rp,
                                                                            ci, v);
        else
            row_sort_kernel<64, 4, T><<<(n + 3) / 4, 256, 0, c->stream>>>(n, trp, tci, tv, place, rp,
                                                                          ci, v);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    int transpose_f64(lal_context* c, int m, int n, int nnz, const int* rp, const int* ci,
                      const double* v, int* trp, int* tci, double* tv, arena* a)
    {
        return transpose_t<double>(c, m, n, nnz, rp, ci, v, trp, tci, tv, a);
    }

    // The symbolic pass: row_ptr of C, its entry count, and in `num` the plan
    // of the numeric pass over it (its bin counts come with the entry count).
    static int symbolic(lal_context* c, int m, int n, const int* arp, const int* aci,
                        const int* brp, const int* bci, int* crp, int* nnz_c, int g, int l,
                        long nnz_a, spgemm_plan& num, temps& tmp, arena* a)
    {
        if(m <= 0)
        {
            LAL_HIP(hipMemsetAsync(crp, 0, sizeof(int), c->stream));
            *nnz_c = 0;
            return LAL_OK;
        }
        spgemm_plan P;
        P.g = g;
        P.l = l;
        LAL_TRY(count_products(c, m, arp, aci, brp, nnz_a, P, tmp));
        LAL_TRY(plan_count(c, m, n, nullptr, false, P, tmp, crp, false, nullptr, a));
        LAL_TRY(plan_rows(c, m, n, nullptr, false, P, tmp));
        LAL_TRY(run_plan<false>(c, P, arp, aci, nullptr, brp, bci, nullptr, nullptr, crp,
                                nullptr));
        num.g = g;
        num.l = l;
        return plan_count(c, m, n, crp, true, num, tmp, nullptr, true, nnz_c, a);
    }

    int csrgemm_nnz(lal_context* c, int m, int k, int n, const int* arp, const int* aci,
                    const int* brp, const int* bci, int* crp, int* nnz_c, long nnz_a, long nnz_b)
    {
        temps       tmp(c, nullptr);
        spgemm_plan num;
        return symbolic(c, m, n, arp, aci, brp, bci, crp, nnz_c, lanes_for(m > 0 ? nnz_a / m : 0),
                        lanes_for(k > 0 ? nnz_b / k : 0), nnz_a, num, tmp, nullptr);
    }

    int csrgemm_solve_f64(lal_context* c, int m, int k, int n, const int* arp, const int* aci,
                          const double* av, const int* brp, const int* bci, const double* bv,
                          const int* crp, int* cci, double* cv, long nnz_a, long nnz_b)
    {
        temps       tmp(c, nullptr);
        spgemm_plan P;
        P.g = lanes_for(m > 0 ? nnz_a / m : 0);
        P.l = lanes_for(k > 0 ? nnz_b / k : 0);
        LAL_TRY(plan_count(c, m, n, const_cast<int*>(crp), true, P, tmp, nullptr, false, nullptr,
                           nullptr));
        LAL_TRY(plan_rows(c, m, n, crp, true, P, tmp));
        LAL_TRY(run_plan<true>(c, P, arp, aci, av, brp, bci, bv, crp, cci, cv));
        int bad = 0;
        LAL_TRY(read_ints(c, c->d_flag, 1, &bad, true));
        if(bad)
        {
            set_last_error("csrgemm_solve: row_ptr of C does not match the product's pattern");
            return LAL_ERR_INVALID;
        }
        return LAL_OK;
    }

    // C = A B for a hierarchy build: C's arrays (nnz entries, m + 1 row
    // pointers) lie in `mem`, the work arrays in `work`.  The operands are the
    // build's own, so the numeric pass's row check cannot fail and is not
    // waited for.
    int product(lal_context* c, int m, int k, int n, int nnz_a, const int* arp, const int* aci,
                const double* av, int nnz_b, const int* brp, const int* bci, const double* bv,
                int** crp, int** cci, double** cv, int* nnz_c, arena* mem, arena* work)
    {
        temps       tmp(c, work);
        spgemm_plan num;
        LAL_TRY(mem->get(crp, (size_t)m + 1));
        LAL_TRY(symbolic(c, m, n, arp, aci, brp, bci, *crp, nnz_c,
                         lanes_for(m > 0 ? nnz_a / m : 0), lanes_for(k > 0 ? nnz_b / k : 0),
                         nnz_a, num, tmp, work));
        LAL_TRY(mem->get(cci, *nnz_c));
        LAL_TRY(mem->get(cv, *nnz_c));
        LAL_TRY(plan_rows(c, m, n, *crp, true, num, tmp));
        return run_plan<true>(c, num, arp, aci, av, brp, bci, bv, *crp, *cci, *cv);
    }
}

namespace
{
    // flag = 1 when a row of B holds a column index twice.  Strictly
    // ascending rows (the usual case) take one pass; other rows compare every
    // pair.
    __global__ void __launch_bounds__(256)
        dup_cols_kernel(int k, const int* __restrict__ brp, const int* __restrict__ bci,
                        int* __restrict__ flag)
    {
        const int row = blockIdx.x * 256 + threadIdx.x;
        if(row >= k)
            return;
        const int rs = brp[row], re = brp[row + 1];
        bool      ascending = true;
        for(int p = rs + 1; p < re && ascending; p++)
            ascending = bci[p] > bci[p - 1];
        if(ascending)
            return;
        for(int p = rs + 1; p < re; p++)
            for(int q = rs; q < p; q++)
                if(bci[q] == bci[p])
                {
                    atomicOr(flag, 1);
                    return;
                }
    }

    // Validates the operands of the C ABI products: column indices of A in
    // [0, k) and of B in [0, n), and no column index repeated within a row of
    // B (the hash pass folds each product into one slot per column, so two
    // lanes meeting the same column of one B row would race; such a matrix is
    // refused rather than summed).
    int check_product_operands(lal_context* c, int k, int n, int nnz_A, const int* aci,
                               int nnz_B, const int* brp, const int* bci)
    {
        // three flags, read together
        LAL_TRY(lal::raise_bad_columns(c, nnz_A, k, aci, c->d_flag));
        LAL_TRY(lal::raise_bad_columns(c, nnz_B, n, bci, c->d_flag + 1));
        if(k > 0 && nnz_B > 0)
        {
            dup_cols_kernel<<<lal::grid_for(k, 256), 256, 0, c->stream>>>(k, brp, bci,
                                                                          c->d_flag + 2);
            LAL_LAUNCHED();
        }
        int bad[3];
        LAL_TRY(lal::read_ints(c, c->d_flag, 3, bad, true));
        if(bad[0] || bad[1])
        {
            lal::set_last_error("column index outside [0, n)");
            return LAL_ERR_INVALID;
        }
        if(bad[2])
        {
            lal::set_last_error("csrgemm: a row of B repeats a column index");
            return LAL_ERR_UNSUPPORTED;
        }
        return LAL_OK;
    }
}

extern "C" int lal_transpose_f64(lal_handle c, int m, int n, int nnz, const int* rp,
                                 const int* ci, const double* v, int* trp, int* tci, double* tv)
{
    LAL_REQUIRE(c != nullptr && m >= 0 && n >= 0 && nnz >= 0 && trp != nullptr);
    LAL_REQUIRE(nnz == 0 || (rp && ci && v && tci && tv));
    return lal::transpose_f64(c, m, n, nnz, rp, ci, v, trp, tci, tv, nullptr);
}

extern "C" int lal_transpose_f32(lal_handle c, int m, int n, int nnz, const int* rp,
                                 const int* ci, const float* v, int* trp, int* tci, float* tv)
{
    LAL_REQUIRE(c != nullptr && m >= 0 && n >= 0 && nnz >= 0 && trp != nullptr);
    LAL_REQUIRE(nnz == 0 || (rp && ci && v && tci && tv));
    return lal::transpose_t<float>(c, m, n, nnz, rp, ci, v, trp, tci, tv, nullptr);
}

extern "C" int lal_csrgemm_nnz(lal_handle c, int m, int k, int n, int nnz_A, const int* arp,
                               const int* aci, int nnz_B, const int* brp, const int* bci,
                               int* crp, int* nnz_C)
{
    LAL_REQUIRE(c != nullptr && m >= 0 && k >= 0 && n >= 0 && nnz_A >= 0 && nnz_B >= 0);
    LAL_REQUIRE(crp != nullptr && nnz_C != nullptr && arp != nullptr && brp != nullptr);
    LAL_REQUIRE((nnz_A == 0 || aci) && (nnz_B == 0 || bci));
    LAL_TRY(check_product_operands(c, k, n, nnz_A, aci, nnz_B, brp, bci));
    return lal::csrgemm_nnz(c, m, k, n, arp, aci, brp, bci, crp, nnz_C, nnz_A, nnz_B);
}

extern "C" int lal_csrgemm_solve_f64(lal_handle c, int m, int k, int n, int nnz_A,
                                     const int* arp, const int* aci, const double* av,
                                     int nnz_B, const int* brp, const int* bci,
                                     const double* bv, const int* crp, int* cci, double* cv)
{
    LAL_REQUIRE(c != nullptr && m >= 0 && k >= 0 && n >= 0 && nnz_A >= 0 && nnz_B >= 0);
    LAL_REQUIRE(crp != nullptr && arp != nullptr && brp != nullptr);
    LAL_REQUIRE((nnz_A == 0 || (aci && av)) && (nnz_B == 0 || (bci && bv)));
    LAL_TRY(check_product_operands(c, k, n, nnz_A, aci, nnz_B, brp, bci));
    return lal::csrgemm_solve_f64(c, m, k, n, arp, aci, av, brp, bci, bv, crp, cci, cv, nnz_A,
                                  nnz_B);
}
