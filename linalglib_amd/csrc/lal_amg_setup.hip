// SA-AMG setup kernels: strength of connection, PMIS aggregation and the
// smoothed prolongator.
//
// Each decision and each floating-point value is formed by the same
// operations in the same order as the host path -- a lane walking its row in
// CSR order, or a group of lanes whose reductions keep the CSR order (entry
// positions as tie-breaks, folds taken lane by lane in entry order):
//   strength     backend/host/host_amg_strength.cpp:33-70
//   PMIS         backend/host/host_amg_aggregation.cpp:32-221 driven as
//                iterative_solvers/amg/amg_aggregation.cpp:106-215
//   prolongator  iterative_solvers/amg/saamg.cpp:51-207
// The library is built with -ffp-contract=off, and HIP's double sqrt and
// division are correctly rounded, so the results are bit-identical.
#include "lal_internal.h"

#include <algorithm>
#include <climits>

namespace
{
    __device__ __forceinline__ int hash1(unsigned x)
    {
        x = ((x >> 16) ^ x) * 0x45d9f3bu;
        x = ((x >> 16) ^ x) * 0x45d9f3bu;
        x = (x >> 16) ^ x;
        return (int)(x / 2);
    }

    __global__ void __launch_bounds__(256)
        pmis_init_kernel(int m, const int* __restrict__ rp, const int* __restrict__ conn,
                         int* __restrict__ state, int* __restrict__ hash)
    {
        int i = blockIdx.x * 256 + threadIdx.x;
        if(i >= m)
            return;
        int s = -2;
        for(int j = rp[i]; j < rp[i + 1]; j++)
            if(conn[j] == 1)
            {
                s = 0;
                break;
            }
        state[i] = s;
        hash[i]  = hash1((unsigned)i);
    }

    // Candidate (s, h, r) replaces the running maximum when its state is
    // strictly greater, or equal with a strictly greater hash.
    __device__ __forceinline__ void lex_max(int& ms, int& mh, int& mr, int s, int h, int r)
    {
        if(s > ms || (s == ms && h > mh))
        {
            ms = s;
            mh = h;
            mr = r;
        }
    }

    // The C ABI's single steps, a lane per row: a decided row's max_state is
    // left alone, as the reference's kernel does.
    __global__ void __launch_bounds__(256)
        pmis_round_kernel(int m, const int* __restrict__ rp, const int* __restrict__ ci,
                          const int* __restrict__ conn, const int* __restrict__ state,
                          const int* __restrict__ hash, int64_t* __restrict__ agg,
                          int* __restrict__ max_state, int* __restrict__ incomplete)
    {
        int i = blockIdx.x * 256 + threadIdx.x;
        if(i >= m)
            return;
        const int si = state[i];
        if(si != 0)
            return; // only undecided rows change anything
        int ms = si, mh = hash[i], mr = i;
        for(int j = rp[i]; j < rp[i + 1]; j++)
            if(conn[j] == 1)
            {
                int c = ci[j];
                lex_max(ms, mh, mr, state[c], hash[c], c);
            }
        const int r2 = mr;
        for(int j = rp[r2]; j < rp[r2 + 1]; j++)
            if(conn[j] == 1)
            {
                int c = ci[j];
                lex_max(ms, mh, mr, state[c], hash[c], c);
            }
        if(mr == i)
        {
            max_state[i] = 1;
            agg[i]       = 1;
        }
        else if(ms == 1)
        {
            max_state[i] = -1;
            agg[i]       = 0;
        }
        else
            *incomplete = 1;
    }

    __global__ void __launch_bounds__(256)
        pmis_join_kernel(int m, const int* __restrict__ rp, const int* __restrict__ ci,
                         const int* __restrict__ conn, const int* __restrict__ state,
                         int64_t* __restrict__ agg, int* __restrict__ max_state)
    {
        int i = blockIdx.x * 256 + threadIdx.x;
        if(i >= m)
            return;
        const int si = state[i];
        if(si == -1)
        {
            for(int j = rp[i]; j < rp[i + 1]; j++)
                if(conn[j] == 1)
                {
                    int c = ci[j];
                    if(state[c] == 1)
                    {
                        // c has state 1 in the snapshot, so its aggregate is
                        // not written during this pass
                        agg[i]       = agg[c];
                        max_state[i] = 1;
                        break;
                    }
                }
        }
        else if(si == -2)
            agg[i] = -2;
    }

    __device__ __forceinline__ bool p_candidate(int i, int c, int cn)
    {
        return c == i || cn == 1;
    }
}

namespace
{
    // The prolongator P = (I - relax D^-1 A_F) T (saamg.cpp:51-207) with G lanes
    // per row (setup_row_lanes).  Row i's entries
    // are its candidates' distinct aggregates >= 0 (the diagonal and the
    // strong neighbours) in ascending order, each the CSR-order fold of its
    // contributions from the first one, with the weak couplings lumped into
    // the diagonal.  The next aggregate in ascending order is a group-wide
    // minimum, and every fold runs over the lanes in entry order.
    //
    // A row's candidates stay in registers, PROLONG_KEEP entries per lane: one
    // read of the row, then every output column is a group minimum and a fold
    // over registers.  The fills of a 121^3 diffusion hierarchy take 0.64 ms;
    // rescanning the row from memory for every column (rows beyond
    // G * PROLONG_KEEP entries still do) they took 1.77.
    constexpr int PROLONG_KEEP = 4;

    template <int G>
    __device__ __forceinline__ int group_min(int v)
    {
        return lal::group_fold<G>(v, [](int a, int b) { return min(a, b); });
    }

    template <int G>
    __device__ __forceinline__ int group_max(int v)
    {
        return lal::group_fold<G>(v, [](int a, int b) { return max(a, b); });
    }

    // Aggregate of entry j's column when it is a candidate of row i (aggregate
    // ids are below the row count, so 32 bits hold them); INT_MAX otherwise.
    __device__ __forceinline__ int candidate_aggregate(int i, int c, int cn,
                                                       const int64_t* __restrict__ agg)
    {
        if(!p_candidate(i, c, cn))
            return INT_MAX;
        const int64_t a = agg[c];
        return a >= 0 ? (int)a : INT_MAX;
    }

    // v of lane t of the group that starts at lane gb (t group-uniform; in a
    // whole wavefront it is a scalar read).
    template <int G, typename V>
    __device__ __forceinline__ V group_lane(V v, int gb, int t)
    {
        if constexpr(G == 64)
            return lal::wave_lane(v, __builtin_amdgcn_readfirstlane(t));
        else
            return __shfl(v, gb + t, 64);
    }

    // Smallest aggregate id above `last` among the row's candidates (INT_MAX
    // when there is none); group-uniform.  key: the lane's first PROLONG_KEEP
    // entries; entries beyond them come from memory.
    // (CI, CN: how a caller holds columns and connections)
    template <int G, typename CI, typename CN>
    __device__ __forceinline__ int next_aggregate(int i, int rs, int re, int gl, bool more,
                                                  const int (&key)[PROLONG_KEEP],
                                                  const CI* __restrict__ ci,
                                                  const CN* __restrict__ conn,
                                                  const int64_t* __restrict__ agg, int last)
    {
        int best = INT_MAX;
#pragma unroll
        for(int u = 0; u < PROLONG_KEEP; u++)
            if(key[u] > last && key[u] < best)
                best = key[u];
        if(more)
            for(int j = rs + G * PROLONG_KEEP + gl; j < re; j += G)
            {
                const int a = candidate_aggregate(i, ci[j], conn[j], agg);
                if(a > last && a < best)
                    best = a;
            }
        return group_min<G>(best);
    }

    // Entries of row i of P (group-uniform).
    template <int G, typename CI, typename CN>
    __device__ __forceinline__ int prolong_count_row(int i, int gl, const int* __restrict__ rp,
                                                     const CI* __restrict__ ci,
                                                     const CN* __restrict__ conn,
                                                     const int64_t* __restrict__ agg)
    {
        const int rs = rp[i], re = rp[i + 1];
        int       key[PROLONG_KEEP];
#pragma unroll
        for(int u = 0; u < PROLONG_KEEP; u++)
        {
            const int j = rs + u * G + gl;
            key[u]      = j < re ? candidate_aggregate(i, ci[j], conn[j], agg) : INT_MAX;
        }
        const bool more = re - rs > G * PROLONG_KEEP;
        int        k    = 0;
        int        last = -1;
        for(;;)
        {
            const int best = next_aggregate<G>(i, rs, re, gl, more, key, ci, conn, agg, last);
            if(best == INT_MAX)
                break;
            k++;
            last = best;
        }
        return k;
    }

    // f(row, lane) by the whole wavefront, for every row of its groups that holds
    // more entries than a group's registers (`len`, -1: no row).  Such a row is read
    // again for every output column, and the lanes per row follow the mean length.
    // Power law, 5000 rows of up to 2500 entries, 28 on average: counts 4.1 ms with
    // a wavefront for every row, 14.0 with 16 lanes, 3.5 so; fills 9.5, 36.3, 9.2.
    // 400,000 rows of up to 3000, 8 lanes for the others: 265 -> 36 and 690 -> 88 ms.
    template <int G, typename F>
    __device__ __forceinline__ void long_rows(int i, int len, F f)
    {
        if constexpr(G < 64)
        {
            const int lane = (int)threadIdx.x & 63;
            for(unsigned long long todo = __ballot(lane % G == 0 && len > G * PROLONG_KEEP);
                todo != 0; todo &= todo - 1)
                f(__builtin_amdgcn_readlane(i, __ffsll((long long)todo) - 1), lane);
        }
    }

    template <int G>
    __global__ void __launch_bounds__(256)
        prolong_count_group_kernel(int m, const int* __restrict__ rp, const int* __restrict__ ci,
                                   const int* __restrict__ conn, const int64_t* __restrict__ agg,
                                   int* __restrict__ count)
    {
        const int gl  = (int)threadIdx.x % G;
        const int i   = blockIdx.x * (256 / G) + (int)threadIdx.x / G;
        const int len = i < m ? rp[i + 1] - rp[i] : -1;
        if(i <= m && (G == 64 || len <= G * PROLONG_KEEP))
        {
            const int k = i < m ? prolong_count_row<G>(i, gl, rp, ci, conn, agg) : 0;
            if(gl == 0)
                count[i] = k;
        }
        long_rows<G>(i, len, [&](int row, int lane) {
            const int k = prolong_count_row<64>(row, lane, rp, ci, conn, agg);
            if(lane == 0)
                count[row] = k;
        });
    }

    // Row i of P into pci/pv[p0 .. p1).
    template <int G, typename CI, typename CN>
    __device__ __forceinline__ void
        prolong_fill_row(int i, int gl, const int* __restrict__ rp, const CI* __restrict__ ci,
                         const double* __restrict__ val, const CN* __restrict__ conn,
                         const int64_t* __restrict__ agg, double relax, int p0, int p1,
                         int* __restrict__ pci, double* __restrict__ pv)
    {
        const int gb = ((int)threadIdx.x & 63) - gl; // the group's first lane
        const int rs = rp[i], re = rp[i + 1];
        int       key[PROLONG_KEEP];
        double    v[PROLONG_KEEP];
        int       kind[PROLONG_KEEP]; // 1: the diagonal, 2: weak, 0: strong or none
#pragma unroll
        for(int u = 0; u < PROLONG_KEEP; u++)
        {
            const int j = rs + u * G + gl;
            key[u]      = INT_MAX;
            v[u]        = 0.0;
            kind[u]     = 0;
            if(j < re)
            {
                const int c = ci[j], cn = conn[j];
                v[u]    = val[j];
                kind[u] = c == i ? 1 : cn == 0 ? 2 : 0;
                key[u]  = candidate_aggregate(i, c, cn, agg);
            }
        }
        const bool more = re - rs > G * PROLONG_KEEP;
        // a_ii minus the weak couplings, summed in CSR order
        double diagonal = 0.0;
        auto   lump     = [&](int kd, double vv) {
            unsigned long long mask = __ballot(kd != 0) >> gb;
            if(G < 64)
                mask &= (1ull << (G % 64)) - 1ull;
            while(mask)
            {
                const int    t  = __ffsll((long long)mask) - 1;
                const int    kt = group_lane<G>(kd, gb, t);
                const double vt = group_lane<G>(vv, gb, t);
                mask &= mask - 1;
                diagonal = kt == 1 ? diagonal + vt : diagonal - vt;
            }
        };
#pragma unroll
        for(int u = 0; u < PROLONG_KEEP; u++)
            lump(kind[u], v[u]);
        if(more)
            for(int j0 = rs + G * PROLONG_KEEP; j0 < re; j0 += G)
            {
                const int j  = j0 + gl;
                int       kd = 0;
                double    vv = 0.0;
                if(j < re)
                {
                    const int c = ci[j];
                    kd          = c == i ? 1 : conn[j] == 0 ? 2 : 0;
                    vv          = val[j];
                }
                lump(kd, vv);
            }
        const double invd = 1.0 / diagonal;
        auto smoothed = [&](bool diag, double a) { return diag ? 1.0 - relax : -relax * invd * a; };
#pragma unroll
        for(int u = 0; u < PROLONG_KEEP; u++)
            v[u] = smoothed(kind[u] == 1, v[u]);
        int last = -1;
        for(int out = p0; out < p1; out++)
        {
            const int best = next_aggregate<G>(i, rs, re, gl, more, key, ci, conn, agg, last);
            bool      first = true;
            double    acc   = 0.0;
            auto      fold  = [&](bool match, double value) {
                unsigned long long mask = __ballot(match) >> gb;
                if(G < 64)
                    mask &= (1ull << (G % 64)) - 1ull;
                while(mask)
                {
                    const int    t  = __ffsll((long long)mask) - 1;
                    const double vt = group_lane<G>(value, gb, t);
                    mask &= mask - 1;
                    acc   = first ? vt : acc + vt;
                    first = false;
                }
            };
#pragma unroll
            for(int u = 0; u < PROLONG_KEEP; u++)
                fold(key[u] == best, v[u]);
            if(more)
                for(int j0 = rs + G * PROLONG_KEEP; j0 < re; j0 += G)
                {
                    const int j     = j0 + gl;
                    bool      match = false;
                    double    value = 0.0;
                    if(j < re)
                    {
                        const int c = ci[j];
                        if(candidate_aggregate(i, c, conn[j], agg) == best)
                        {
                            match = true;
                            value = smoothed(c == i, val[j]);
                        }
                    }
                    fold(match, value);
                }
            if(gl == 0)
            {
                pci[out] = best;
                pv[out]  = acc;
            }
            last = best;
        }
    }

    template <int G>
    __global__ void __launch_bounds__(256)
        prolong_fill_group_kernel(int m, const int* __restrict__ rp, const int* __restrict__ ci,
                                  const double* __restrict__ val, const int* __restrict__ conn,
                                  const int64_t* __restrict__ agg, double relax,
                                  const int* __restrict__ prp, int* __restrict__ pci,
                                  double* __restrict__ pv)
    {
        const int gl  = (int)threadIdx.x % G;
        const int i   = blockIdx.x * (256 / G) + (int)threadIdx.x / G;
        const int len = i < m ? rp[i + 1] - rp[i] : -1;
        if(i < m && (G == 64 || len <= G * PROLONG_KEEP))
            prolong_fill_row<G>(i, gl, rp, ci, val, conn, agg, relax, prp[i], prp[i + 1], pci, pv);
        long_rows<G>(i, len, [&](int row, int lane) {
            prolong_fill_row<64>(row, lane, rp, ci, val, conn, agg, relax, prp[row], prp[row + 1],
                                 pci, pv);
        });
    }
}

namespace
{
    // Strength, the diagonal and the PMIS passes with G lanes per row (8,
    // 16 or 64, 256 / G rows per workgroup): a lane walking a row alone is a
    // chain of dependent, strided loads.  Each lane takes the row's entries
    // j = rs + gl, rs + gl + G, ... in order; every per-row result the
    // thread-per-row kernels form in CSR order -- the first (or last) match,
    // a lexicographic maximum that keeps its first occurrence -- is the
    // group's reduction with the entry position as the tie-break, so the
    // results are bit for bit the same.
    template <int G>
    __device__ __forceinline__ int group_row(int& gl)
    {
        gl = (int)threadIdx.x % G;
        return blockIdx.x * (256 / G) + (int)threadIdx.x / G;
    }

    // d[i] = the row's first diagonal entry (0 when it has none)
    template <int G>
    __global__ void __launch_bounds__(256)
        diagonal_group_kernel(int m, const int* __restrict__ rp, const int* __restrict__ ci,
                              const double* __restrict__ val, double* __restrict__ d)
    {
        int       gl;
        const int i = group_row<G>(gl);
        if(i >= m)
            return;
        const int rs = rp[i], re = rp[i + 1];
        int       first = INT_MAX;
        for(int j = rs + gl; j < re; j += G)
            if(ci[j] == i)
            {
                first = j;
                break;
            }
        first = group_min<G>(first);
        if(gl == 0 && first != INT_MAX)
            d[i] = val[first];
    }

    template <int G>
    __global__ void __launch_bounds__(256)
        strength_group_kernel(int m, const int* __restrict__ rp, const int* __restrict__ ci,
                              const double* __restrict__ val, const double* __restrict__ d,
                              double eps, int* __restrict__ conn)
    {
        int       gl;
        const int i = group_row<G>(gl);
        if(i >= m)
            return;
        const double di = fabs(d[i]);
        for(int j = rp[i] + gl; j < rp[i + 1]; j += G)
        {
            int    c = ci[j];
            double v = val[j];
            conn[j]  = (c != i) && (fabs(v) >= eps * sqrt(di * fabs(d[c])));
        }
    }

    template <int G>
    __global__ void __launch_bounds__(256)
        pmis_init_group_kernel(int m, const int* __restrict__ rp, const int* __restrict__ conn,
                               int* __restrict__ state, int* __restrict__ hash)
    {
        int       gl;
        const int i = group_row<G>(gl);
        if(i >= m)
            return;
        int strong = 0;
        for(int j = rp[i] + gl; j < rp[i + 1] && !strong; j += G)
            strong = conn[j] == 1;
        strong = group_max<G>(strong);
        if(gl == 0)
        {
            state[i] = strong ? 0 : -2;
            hash[i]  = hash1((unsigned)i);
        }
    }

    // A PMIS candidate: state, hash, node, and its position in the scan.
    struct pmis_cand
    {
        int s, h, r, pos;
    };

    // b replaces a when (s, h) is lexicographically greater, or equal and
    // earlier in the scan.
    __device__ __forceinline__ void pmis_take(pmis_cand& a, const pmis_cand& b)
    {
        if(b.s > a.s || (b.s == a.s && (b.h > a.h || (b.h == a.h && b.pos < a.pos))))
            a = b;
    }

    // The best strong neighbour of row `row` across the group: each lane keeps
    // the first maximum of its entries, the group the earliest of the lanes'.
    template <int G, typename CI, typename CN>
    __device__ __forceinline__ pmis_cand pmis_scan(int row, int gl, const int* __restrict__ rp,
                                                   const CI* __restrict__ ci,
                                                   const CN* __restrict__ conn,
                                                   const int* __restrict__ state,
                                                   const int* __restrict__ hash)
    {
        pmis_cand best{INT_MIN, INT_MIN, -1, INT_MAX};
        const int rs = rp[row], re = rp[row + 1];
        for(int j = rs + gl; j < re; j += G)
            if(conn[j] == 1)
            {
                const int c = ci[j];
                const int sc = state[c], hc = hash[c];
                if(sc > best.s || (sc == best.s && hc > best.h))
                    best = pmis_cand{sc, hc, c, j - rs};
            }
        const auto take = [&](auto at) {
            pmis_take(best, pmis_cand{at(best.s), at(best.h), at(best.r), at(best.pos)});
        };
        take([](int v) { return lal::partner<0>(v); });
        take([](int v) { return lal::partner<1>(v); });
        take([](int v) { return lal::partner<2>(v); });
        if(G >= 16)
            take([](int v) { return lal::partner<3>(v); });
        if(G == 64)
        {
            const pmis_cand mine = best;
            const auto      row  = [&](int t) {
                return pmis_cand{
                    __builtin_amdgcn_readlane(mine.s, t), __builtin_amdgcn_readlane(mine.h, t),
                    __builtin_amdgcn_readlane(mine.r, t), __builtin_amdgcn_readlane(mine.pos, t)};
            };
            best = row(0);
            pmis_take(best, row(16));
            pmis_take(best, row(32));
            pmis_take(best, row(48));
        }
        return best;
    }

    // pmis_round_kernel with G lanes per row: the running maximum starts at
    // the row itself, takes the row's strong neighbours in order, then the
    // strong neighbours of the row that maximum names.
    // Every row's state goes to max_state, decided or not, so that the rounds
    // alternate two buffers.
    template <int G, typename CI, typename CN>
    __device__ __forceinline__ void
        pmis_round_row(int i, int gl, const int* __restrict__ rp, const CI* __restrict__ ci,
                       const CN* __restrict__ conn, const int* __restrict__ state,
                       const int* __restrict__ hash, int64_t* __restrict__ agg,
                       int* __restrict__ max_state, int* __restrict__ incomplete)
    {
        const int si = state[i];
        if(si != 0)
        {
            if(gl == 0)
                max_state[i] = si;
            return; // only undecided rows change anything
        }
        // the row itself precedes its neighbours, so it wins a tie
        pmis_cand run{si, hash[i], i, -1};
        pmis_cand c1 = pmis_scan<G>(i, gl, rp, ci, conn, state, hash);
        if(c1.s > run.s || (c1.s == run.s && c1.h > run.h))
            run = c1;
        // the second row's entries all follow the first scan's
        pmis_cand c2 = pmis_scan<G>(run.r, gl, rp, ci, conn, state, hash);
        if(c2.s > run.s || (c2.s == run.s && c2.h > run.h))
            run = c2;
        if(gl != 0)
            return;
        if(run.r == i)
        {
            max_state[i] = 1;
            agg[i]       = 1;
        }
        else if(run.s == 1)
        {
            max_state[i] = -1;
            agg[i]       = 0;
        }
        else
            *incomplete = 1;
    }

    template <int G>
    __global__ void __launch_bounds__(256)
        pmis_round_group_kernel(int m, const int* __restrict__ rp, const int* __restrict__ ci,
                                const int* __restrict__ conn, const int* __restrict__ state,
                                const int* __restrict__ hash, int64_t* __restrict__ agg,
                                int* __restrict__ max_state, int* __restrict__ incomplete)
    {
        int       gl;
        const int i = group_row<G>(gl);
        if(i < m)
            pmis_round_row<G>(i, gl, rp, ci, conn, state, hash, agg, max_state, incomplete);
    }

    template <int G, typename CI, typename CN>
    __device__ __forceinline__ void
        pmis_join_row(int i, int gl, const int* __restrict__ rp, const CI* __restrict__ ci,
                      const CN* __restrict__ conn, const int* __restrict__ state, int64_t* agg,
                      int* __restrict__ max_state)
    {
        const int si = state[i];
        if(gl == 0)
            max_state[i] = si;
        if(si == -1)
        {
            // the first strong neighbour (in CSR order) with state 1
            int first = INT_MAX;
            for(int j = rp[i] + gl; j < rp[i + 1]; j += G)
                if(conn[j] == 1 && state[ci[j]] == 1)
                {
                    first = j;
                    break;
                }
            first = group_min<G>(first);
            if(gl == 0 && first != INT_MAX)
            {
                // c has state 1 in the snapshot, so its aggregate is not
                // written during this pass
                agg[i]       = agg[ci[first]];
                max_state[i] = 1;
            }
        }
        else if(si == -2 && gl == 0)
            agg[i] = -2;
    }

    template <int G>
    __global__ void __launch_bounds__(256)
        pmis_join_group_kernel(int m, const int* __restrict__ rp, const int* __restrict__ ci,
                               const int* __restrict__ conn, const int* __restrict__ state,
                               int64_t* __restrict__ agg, int* __restrict__ max_state)
    {
        int       gl;
        const int i = group_row<G>(gl);
        if(i < m)
            pmis_join_row<G>(i, gl, rp, ci, conn, state, agg, max_state);
    }

    // A level from its operator to P and R = P^T in one workgroup.
    struct small_level
    {
        int           m, nnz;
        const int *   rp, *ci;
        const double* v;
        double        eps, relax;
        bool          unsmoothed;
        int*          place; // scratch, one per entry of P: its place in R's row,
        int*          tci;   // and R's entries before they are in order
        double*       tv;
        int *         prp, *pci, *rrp, *rci;
        double *      pv, *rv;
    };
    constexpr int SMALL_THREADS = 1024;
    constexpr int SMALL_ROWS    = 1024; // (columns fit 16 bits)
    constexpr int SMALL_NNZ     = 8192;

    // Exclusive scan over the workgroup, one value per lane.
    __device__ __forceinline__ int small_scan(int v, int* total)
    {
        __shared__ int s_w[SMALL_THREADS / 64];
        const int      lane = (int)threadIdx.x & 63, wid = (int)threadIdx.x >> 6;
        int            inc  = v;
#pragma unroll
        for(int o = 1; o < 64; o <<= 1)
        {
            const int q = __shfl_up(inc, o, 64);
            inc += lane >= o ? q : 0;
        }
        __syncthreads();
        if(lane == 63)
            s_w[wid] = inc;
        __syncthreads();
        int at = inc - v, all = 0;
        for(int w = 0; w < SMALL_THREADS / 64; w++)
        {
            at += w < wid ? s_w[w] : 0;
            all += s_w[w];
        }
        *total = all;
        return at;
    }

    // The steps of the passes above and of the transpose, row by row with the
    // same functions, so the results are theirs bit for bit; states, hashes and
    // aggregates lie in LDS.  Level after level these were 27 launches of a few
    // microseconds and two waits for the host: the time of a small hierarchy.
    // 25^3 diffusion, levels of 84, 12 and 3 rows, with the products' plans in
    // one launch too: 318 launches and 2.36 ms -> 207 and 2.12.  One workgroup is
    // slower per row than the chip (84 rows of 84 entries: 112 us), so a level
    // comes here up to where its launches would take about as long.
    // The note: columns of P, entries of P.
    template <int G>
    __global__ void __launch_bounds__(SMALL_THREADS)
        small_level_kernel(small_level a, int* note, unsigned seq)
    {
        constexpr int             NG = SMALL_THREADS / G;
        __shared__ double         s_d[SMALL_ROWS];
        __shared__ int64_t        s_agg[SMALL_ROWS];
        __shared__ int            s_state[2][SMALL_ROWS], s_hash[SMALL_ROWS], s_cnt[SMALL_ROWS];
        __shared__ int            s_rp[SMALL_ROWS + 1];
        __shared__ unsigned short s_ci[SMALL_NNZ];
        __shared__ unsigned char  s_conn[SMALL_NNZ];
        __shared__ int            s_flag, s_top;
        const int                 tid = (int)threadIdx.x, gl = tid % G, g0 = tid / G, m = a.m;
        if(tid == 0)
        {
            s_top   = -1;
            s_rp[m] = a.nnz;
        }
        if(tid < m)
            s_rp[tid] = a.rp[tid];
        for(int e = tid; e < a.nnz; e += SMALL_THREADS)
            s_ci[e] = (unsigned short)a.ci[e];
        __syncthreads();
        // the row's first diagonal entry (0 when it has none)
        for(int i = g0; i < m; i += NG)
        {
            const int rs = s_rp[i], re = s_rp[i + 1];
            int       first = INT_MAX;
            for(int j = rs + gl; j < re; j += G)
                if(s_ci[j] == i)
                {
                    first = j;
                    break;
                }
            first = group_min<G>(first);
            if(gl == 0)
                s_d[i] = first != INT_MAX ? a.v[first] : 0.0;
        }
        __syncthreads();
        for(int i = g0; i < m; i += NG)
        {
            const double di     = fabs(s_d[i]);
            int          strong = 0;
            for(int j = s_rp[i] + gl; j < s_rp[i + 1]; j += G)
            {
                const int c  = s_ci[j];
                const int on = (c != i) && (fabs(a.v[j]) >= a.eps * sqrt(di * fabs(s_d[c])));
                s_conn[j]    = (unsigned char)on;
                strong |= on;
            }
            strong = group_max<G>(strong);
            if(gl == 0)
            {
                s_state[0][i] = s_state[1][i] = strong ? 0 : -2;
                s_hash[i]                     = hash1((unsigned)i);
                s_agg[i]                      = 0;
            }
        }
        int cur = 0;
        for(int iter = 0; iter < 20; iter++)
        {
            __syncthreads();
            if(tid == 0)
                s_flag = 0;
            __syncthreads();
            for(int i = g0; i < m; i += NG)
                pmis_round_row<G>(i, gl, s_rp, s_ci, s_conn, s_state[cur], s_hash, s_agg,
                                  s_state[cur ^ 1], &s_flag);
            cur ^= 1;
            __syncthreads();
            if(s_flag == 0)
                break;
        }
        int       total = 0;
        const int ahead = small_scan(tid < m ? (int)s_agg[tid] : 0, &total);
        if(tid < m)
            s_agg[tid] = ahead;
        for(int k = 0; k < 2; k++, cur ^= 1)
        {
            __syncthreads();
            for(int i = g0; i < m; i += NG)
                pmis_join_row<G>(i, gl, s_rp, s_ci, s_conn, s_state[cur], s_agg,
                                 s_state[cur ^ 1]);
        }
        __syncthreads();
        // P's row pointer and columns
        for(int i = g0; i < m; i += NG)
        {
            const int k = a.unsmoothed ? s_agg[i] >= 0
                                       : prolong_count_row<G>(i, gl, s_rp, s_ci, s_conn, s_agg);
            if(gl == 0)
                s_cnt[i] = k;
        }
        if(tid < m)
            atomicMax(&s_top, (int)s_agg[tid]);
        __syncthreads();
        int       nnz = 0;
        const int p0  = small_scan(tid < m ? s_cnt[tid] : 0, &nnz);
        if(tid < m)
            a.prp[tid] = p0;
        if(tid == 0)
            a.prp[m] = nnz;
        const int nc = s_top + 1;
        __syncthreads();
        for(int i = g0; i < m; i += NG)
        {
            const int at = a.prp[i], end = a.prp[i + 1];
            if(!a.unsmoothed)
                prolong_fill_row<G>(i, gl, s_rp, s_ci, a.v, s_conn, s_agg, a.relax, at, end, a.pci,
                                    a.pv);
            else if(gl == 0 && s_agg[i] >= 0)
            {
                a.pci[at] = (int)s_agg[i];
                a.pv[at]  = 1.0;
            }
        }
        // R = P^T: places by counting, then every row sorted by rank
        s_cnt[tid] = 0;
        __syncthreads();
        for(int e = tid; e < nnz; e += SMALL_THREADS)
            a.place[e] = atomicAdd(&s_cnt[a.pci[e]], 1);
        __syncthreads();
        int       same = 0;
        const int r0   = small_scan(tid < nc ? s_cnt[tid] : 0, &same);
        if(tid < nc)
            a.rrp[tid] = r0;
        if(tid == 0)
            a.rrp[nc] = nnz;
        __syncthreads();
        for(int i = g0; i < m; i += NG)
            for(int e = a.prp[i] + gl; e < a.prp[i + 1]; e += G)
            {
                const int at = a.rrp[a.pci[e]] + a.place[e];
                a.tci[at]    = i;
                a.tv[at]     = a.pv[e];
            }
        __syncthreads();
        for(int c = g0; c < nc; c += NG)
        {
            const int rs = a.rrp[c], re = a.rrp[c + 1];
            for(int e = rs + gl; e < re; e += G)
            {
                const int row  = a.tci[e];
                int       rank = rs;
                for(int q = rs; q < re; q++)
                    rank += a.tci[q] < row;
                a.rci[rank] = row;
                a.rv[rank]  = a.tv[e];
            }
        }
        if(tid < 64)
            lal::put_note(note, 2, tid == 0 ? nc : nnz, seq);
    }

    __device__ __forceinline__ long long wave_max_i64(long long v)
    {
#pragma unroll
        for(int o = 32; o > 0; o >>= 1)
        {
            const long long t = __shfl_xor(v, o, 64);
            v                 = t > v ? t : v;
        }
        return v;
    }

    // Largest of the workgroup's values, in thread 0.
    __device__ __forceinline__ long long block_max_i64(long long v)
    {
        __shared__ long long s_m[4];
        v = wave_max_i64(v);
        if((threadIdx.x & 63) == 0)
            s_m[threadIdx.x >> 6] = v;
        __syncthreads();
        const long long a = s_m[0] > s_m[1] ? s_m[0] : s_m[1];
        const long long b = s_m[2] > s_m[3] ? s_m[2] : s_m[3];
        return a > b ? a : b;
    }

    __global__ void __launch_bounds__(256)
        max_agg_kernel(int m, const int64_t* __restrict__ agg, long long* __restrict__ part)
    {
        long long v = LLONG_MIN;
        for(int i = blockIdx.x * 256 + threadIdx.x; i < m; i += gridDim.x * 256)
            v = agg[i] > v ? agg[i] : v;
        v = block_max_i64(v);
        if(threadIdx.x == 0)
            part[blockIdx.x] = v;
    }

    // out: {largest of the 256 partials, *nnz}
    __global__ void __launch_bounds__(256)
        max_agg_finish_kernel(const long long* __restrict__ part, const int* __restrict__ nnz,
                              long long* __restrict__ out)
    {
        const long long v = block_max_i64(part[threadIdx.x]);
        if(threadIdx.x == 0)
        {
            out[0] = v;
            out[1] = *nnz;
        }
    }

    // Lanes per row for the row-walking setup passes: 8 for short rows (the
    // finest level's stencil, whose rows a lane alone would read one entry
    // after another, strided), 16 or 64 for the coarse Galerkin levels.
    inline int setup_row_lanes(long nnz, int m)
    {
        const long avg = m > 0 ? nnz / m : 0;
        return avg >= 48 ? 64 : avg >= 12 ? 16 : 8;
    }

    inline int group_grid(int m, int lanes)
    {
        return (int)(((long)m * lanes + 255) / 256);
    }
}

namespace lal
{
    int diagonal_f64(lal_context* c, int m, const int* rp, const int* ci, const double* v,
                     double* d);

    int sa_strength(lal_context* c, int m, int nnz, const int* rp, const int* ci,
                    const double* v, double eps, int* conn, arena* a)
    {
        if(m == 0)
            return LAL_OK;
        temps   tmp(c, a);
        double* d = nullptr;
        LAL_TRY(tmp.get(&d, m));
        LAL_HIP(hipMemsetAsync(d, 0, sizeof(double) * m, c->stream));
        const int lanes = setup_row_lanes(nnz, m);
        const int gg    = group_grid(m, lanes);
#define LAL_LANES(G)                                                                         \
    case G:                                                                                  \
        diagonal_group_kernel<G><<<gg, 256, 0, c->stream>>>(m, rp, ci, v, d);                \
        LAL_LAUNCHED();                                                                      \
        strength_group_kernel<G><<<gg, 256, 0, c->stream>>>(m, rp, ci, v, d, eps, conn);     \
        break;
        switch(lanes)
        {
            LAL_LANES(64)
            LAL_LANES(16)
            LAL_LANES(8)
        }
#undef LAL_LANES
        LAL_LAUNCHED();
        return LAL_OK;
    }

    int pmis_aggregate(lal_context* c, int m, int nnz, const int* rp, const int* ci,
                       const int* conn, int64_t* agg, arena* a)
    {
        if(m == 0)
            return LAL_OK;
        temps tmp(c, a);
        int * state = nullptr, *max_state = nullptr, *hash = nullptr;
        LAL_TRY(tmp.get(&state, m));
        LAL_TRY(tmp.get(&max_state, m));
        LAL_TRY(tmp.get(&hash, m));
        LAL_HIP(hipMemsetAsync(agg, 0, sizeof(int64_t) * m, c->stream));
        const int lanes = setup_row_lanes(nnz, m);
        const int gg    = group_grid(m, lanes);
        if(lanes == 64)
            pmis_init_group_kernel<64><<<gg, 256, 0, c->stream>>>(m, rp, conn, max_state, hash);
        else if(lanes == 16)
            pmis_init_group_kernel<16><<<gg, 256, 0, c->stream>>>(m, rp, conn, max_state, hash);
        else
            pmis_init_group_kernel<8><<<gg, 256, 0, c->stream>>>(m, rp, conn, max_state, hash);
        LAL_LAUNCHED();
        // The reference's loop (amg_aggregation.cpp:106-215): up to 20 rounds,
        // state = max_state before each, stop after the first complete one.
        // Here the rounds alternate between two buffers (the round kernel
        // writes every decided row through, and a row still undecided was
        // undecided in the older buffer too, so it reads 0 there as in the
        // copy), and the host checks after an even number of rounds: a round
        // after a complete one finds no undecided row and changes nothing, so
        // the aggregates are those of the reference's loop.
        // (the first round reads max_state and writes every row of state that
        // it decides; rows it leaves undecided must read 0 there)
        LAL_HIP(hipMemcpyAsync(state, max_state, sizeof(int) * m, hipMemcpyDeviceToDevice,
                               c->stream));
        int* buf[2] = {max_state, state}; // buf[cur]: the latest state
        int  cur    = 0;
        auto round  = [&](int* flag) -> int {
            const int* in  = buf[cur];
            int*       out = buf[cur ^ 1];
            if(lanes == 64)
                pmis_round_group_kernel<64><<<gg, 256, 0, c->stream>>>(m, rp, ci, conn, in, hash,
                                                                       agg, out, flag);
            else if(lanes == 16)
                pmis_round_group_kernel<16><<<gg, 256, 0, c->stream>>>(m, rp, ci, conn, in, hash,
                                                                       agg, out, flag);
            else
                pmis_round_group_kernel<8><<<gg, 256, 0, c->stream>>>(m, rp, ci, conn, in, hash,
                                                                      agg, out, flag);
            LAL_LAUNCHED();
            cur ^= 1;
            return LAL_OK;
        };
        // Six rounds suffice nearly always; a flag per round, read together.
        for(int iter = 0; iter < 20;)
        {
            const int n = iter == 0 ? 6 : 2;
            int       flags[6];
            for(int k = 0; k < n; k++)
                LAL_TRY(round(c->d_flag + k));
            LAL_TRY(read_ints(c, c->d_flag, n, flags, true));
            iter += n;
            if(flags[n - 1] == 0)
                break;
        }
        // (an even number of rounds: the latest state is in max_state again)
        LAL_TRY(scan_i64_dev(c, m, agg, a));
        for(int k = 0; k < 2; k++)
        {
            const int* in  = buf[k];
            int*       out = buf[k ^ 1];
            if(lanes == 64)
                pmis_join_group_kernel<64>
                    <<<gg, 256, 0, c->stream>>>(m, rp, ci, conn, in, agg, out);
            else if(lanes == 16)
                pmis_join_group_kernel<16>
                    <<<gg, 256, 0, c->stream>>>(m, rp, ci, conn, in, agg, out);
            else
                pmis_join_group_kernel<8>
                    <<<gg, 256, 0, c->stream>>>(m, rp, ci, conn, in, agg, out);
            LAL_LAUNCHED();
        }
        return LAL_OK;
    }

    // Levels that small_build takes: at most eight rows for each of the
    // workgroup's lane groups.
    bool small_fits(int m, long nnz)
    {
        return m > 0 && m <= SMALL_ROWS && nnz <= SMALL_NNZ &&
               m * setup_row_lanes(nnz, m) <= 8 * SMALL_THREADS;
    }

    // Strength to R = P^T of one small level.  P's and R's arrays have room for
    // max(m, nnz) entries, R's row pointer for m + 1.
    int small_build(lal_context* c, int m, int nnz, const int* rp, const int* ci, const double* v,
                    double eps, double relax, bool unsmoothed, int* prp, int* pci, double* pv,
                    int* rrp, int* rci, double* rv, int* nnz_P, int* n_c, arena* a)
    {
        LAL_REQUIRE(small_fits(m, nnz));
        temps       tmp(c, a);
        const int   room = std::max(m, nnz);
        small_level L{m,       nnz,     rp,  ci,  v,   eps, relax, unsmoothed, nullptr,
                      nullptr, nullptr, prp, pci, rrp, rci, pv,    rv};
        LAL_TRY(tmp.get(&L.place, room));
        LAL_TRY(tmp.get(&L.tci, room));
        LAL_TRY(tmp.get(&L.tv, room));
        const int      lanes = setup_row_lanes(nnz, m);
        const unsigned seq   = ++c->note_seq;
        auto*          fn    = lanes == 64   ? small_level_kernel<64>
                               : lanes == 16 ? small_level_kernel<16>
                                             : small_level_kernel<8>;
        fn<<<1, SMALL_THREADS, 0, c->stream>>>(L, c->d_note, seq);
        LAL_LAUNCHED();
        int got[2];
        LAL_TRY(take_note(c, seq, 2, got));
        *n_c   = got[0];
        *nnz_P = got[1];
        return LAL_OK;
    }

    // Entries (prp[m]) and columns (the largest aggregate id + 1) of a
    // prolongator whose row pointer has been scanned.
    static int prolongator_size(lal_context* c, int m, const int64_t* agg, const int* prp,
                                int* nnz_P, int* n_c, arena* a)
    {
        constexpr int MAXB = 256;
        temps         tmp(c, a);
        long long*    part = nullptr;
        int           got[3];
        LAL_TRY(tmp.get(&part, MAXB + 2));
        max_agg_kernel<<<MAXB, 256, 0, c->stream>>>(m, agg, part);
        LAL_LAUNCHED();
        max_agg_finish_kernel<<<1, MAXB, 0, c->stream>>>(part, prp + m, part + MAXB);
        LAL_LAUNCHED();
        LAL_TRY(read_ints(c, reinterpret_cast<int*>(part + MAXB), 3, got, false));
        const int64_t mx = (int64_t)(((uint64_t)(uint32_t)got[1] << 32) | (uint32_t)got[0]);
        const int64_t nc = std::max<int64_t>(mx, -1) + 1;
        if(nc > INT_MAX)
            return LAL_ERR_UNSUPPORTED;
        *nnz_P = got[2];
        *n_c   = (int)nc;
        return LAL_OK;
    }

    int sa_prolongator_nnz(lal_context* c, int m, int nnz, const int* rp, const int* ci,
                           const int* conn, const int64_t* agg, int* prp, int* nnz_P,
                           int* n_c, arena* a)
    {
        // count[m] = 0 is written by the group of row m, so m + 1 groups
        const int lanes = setup_row_lanes(nnz, m);
        const int gg    = group_grid(m + 1, lanes);
        if(lanes == 64)
            prolong_count_group_kernel<64><<<gg, 256, 0, c->stream>>>(m, rp, ci, conn, agg, prp);
        else if(lanes == 16)
            prolong_count_group_kernel<16><<<gg, 256, 0, c->stream>>>(m, rp, ci, conn, agg, prp);
        else
            prolong_count_group_kernel<8><<<gg, 256, 0, c->stream>>>(m, rp, ci, conn, agg, prp);
        LAL_LAUNCHED();
        LAL_TRY(scan_i32_dev(c, m + 1, prp, a));
        return prolongator_size(c, m, agg, prp, nnz_P, n_c, a);
    }

    int sa_prolongator_fill(lal_context* c, int m, int nnz, const int* rp, const int* ci,
                            const double* v, const int* conn, const int64_t* agg, double relax,
                            const int* prp, int* pci, double* pv)
    {
        if(m == 0)
            return LAL_OK;
        const int lanes = setup_row_lanes(nnz, m);
        const int gg    = group_grid(m, lanes);
        if(lanes == 64)
            prolong_fill_group_kernel<64><<<gg, 256, 0, c->stream>>>(m, rp, ci, v, conn, agg,
                                                                     relax, prp, pci, pv);
        else if(lanes == 16)
            prolong_fill_group_kernel<16><<<gg, 256, 0, c->stream>>>(m, rp, ci, v, conn, agg,
                                                                     relax, prp, pci, pv);
        else
            prolong_fill_group_kernel<8><<<gg, 256, 0, c->stream>>>(m, rp, ci, v, conn, agg,
                                                                    relax, prp, pci, pv);
        LAL_LAUNCHED();
        return LAL_OK;
    }
}

namespace
{
    // Unsmoothed aggregation (uaamg.cpp:48-123): row i of P holds one entry,
    // 1.0 in column agg[i], when the row was aggregated and nothing otherwise.
    __global__ void __launch_bounds__(256)
        ua_count_kernel(int m, const int64_t* __restrict__ agg, int* __restrict__ prp)
    {
        const int i = blockIdx.x * 256 + threadIdx.x;
        if(i <= m)
            prp[i] = (i < m && agg[i] >= 0) ? 1 : 0;
    }

    __global__ void __launch_bounds__(256)
        ua_fill_kernel(int m, const int64_t* __restrict__ agg, const int* __restrict__ prp,
                       int* __restrict__ pci, double* __restrict__ pv)
    {
        const int i = blockIdx.x * 256 + threadIdx.x;
        if(i < m && agg[i] >= 0)
        {
            pci[prp[i]] = (int)agg[i];
            pv[prp[i]]  = 1.0;
        }
    }
}

namespace lal
{
    int ua_prolongator_nnz(lal_context* c, int m, const int64_t* agg, int* prp, int* nnz_P,
                           int* n_c, arena* a)
    {
        ua_count_kernel<<<grid_for(m + 1, 256), 256, 0, c->stream>>>(m, agg, prp);
        LAL_LAUNCHED();
        LAL_TRY(scan_i32_dev(c, m + 1, prp, a));
        return prolongator_size(c, m, agg, prp, nnz_P, n_c, a);
    }

    int ua_prolongator_fill(lal_context* c, int m, const int64_t* agg, const int* prp, int* pci,
                            double* pv)
    {
        if(m == 0)
            return LAL_OK;
        ua_fill_kernel<<<grid_for(m, 256), 256, 0, c->stream>>>(m, agg, prp, pci, pv);
        LAL_LAUNCHED();
        return LAL_OK;
    }
}

extern "C" int lal_sa_strength_f64(lal_handle c, int m, int nnz, const int* rp, const int* ci,
                                   const double* v, double eps, int* conn)
{
    LAL_REQUIRE(c != nullptr && m >= 0 && nnz >= 0);
    LAL_REQUIRE(m == 0 || (rp && (nnz == 0 || (ci && v && conn))));
    return lal::sa_strength(c, m, nnz, rp, ci, v, eps, conn, nullptr);
}

extern "C" int lal_pmis_aggregate(lal_handle c, int m, int nnz, const int* rp, const int* ci,
                                  const int* conn, int64_t* agg)
{
    LAL_REQUIRE(c != nullptr && m >= 0 && nnz >= 0);
    LAL_REQUIRE(m == 0 || (rp && agg && (nnz == 0 || (ci && conn))));
    return lal::pmis_aggregate(c, m, nnz, rp, ci, conn, agg, nullptr);
}

extern "C" int lal_pmis_init(lal_handle c, int m, int nnz, const int* rp, const int* conn,
                             int* state, int* hash)
{
    LAL_REQUIRE(c != nullptr && m >= 0 && nnz >= 0);
    LAL_REQUIRE(m == 0 || (rp && state && hash && (nnz == 0 || conn)));
    if(m == 0)
        return LAL_OK;
    pmis_init_kernel<<<lal::grid_for(m, 256), 256, 0, c->stream>>>(m, rp, conn, state, hash);
    LAL_LAUNCHED();
    return LAL_OK;
}

extern "C" int lal_pmis_round(lal_handle c, int m, int nnz, const int* rp, const int* ci,
                              const int* conn, const int* state, const int* hash, int64_t* agg,
                              int* max_state, int* complete)
{
    LAL_REQUIRE(c != nullptr && m >= 0 && nnz >= 0 && complete != nullptr);
    LAL_REQUIRE(m == 0 || (rp && state && hash && agg && max_state && (nnz == 0 || (ci && conn))));
    *complete = 1;
    if(m == 0)
        return LAL_OK;
    pmis_round_kernel<<<lal::grid_for(m, 256), 256, 0, c->stream>>>(
        m, rp, ci, conn, state, hash, agg, max_state, c->d_flag);
    LAL_LAUNCHED();
    int undecided = 0;
    LAL_TRY(lal::read_ints(c, c->d_flag, 1, &undecided, true));
    *complete = undecided == 0;
    return LAL_OK;
}

extern "C" int lal_pmis_join(lal_handle c, int m, int nnz, const int* rp, const int* ci,
                             const int* conn, const int* state, int64_t* agg, int* max_state)
{
    LAL_REQUIRE(c != nullptr && m >= 0 && nnz >= 0);
    LAL_REQUIRE(m == 0 || (rp && state && agg && max_state && (nnz == 0 || (ci && conn))));
    if(m == 0)
        return LAL_OK;
    pmis_join_kernel<<<lal::grid_for(m, 256), 256, 0, c->stream>>>(
        m, rp, ci, conn, state, agg, max_state);
    LAL_LAUNCHED();
    return LAL_OK;
}

extern "C" int lal_sa_prolongator_nnz(lal_handle c, int m, int nnz, const int* rp,
                                      const int* ci, const int* conn, const int64_t* agg,
                                      int* prp, int* nnz_P, int* n_c)
{
    LAL_REQUIRE(c != nullptr && m >= 0 && nnz >= 0 && prp && nnz_P && n_c);
    LAL_REQUIRE(m == 0 || (rp && agg && (nnz == 0 || (ci && conn))));
    return lal::sa_prolongator_nnz(c, m, nnz, rp, ci, conn, agg, prp, nnz_P, n_c, nullptr);
}

extern "C" int lal_sa_prolongator_fill_f64(lal_handle c, int m, int nnz, const int* rp,
                                           const int* ci, const double* v, const int* conn,
                                           const int64_t* agg, double relax, const int* prp,
                                           int* pci, double* pv)
{
    LAL_REQUIRE(c != nullptr && m >= 0 && nnz >= 0);
    LAL_REQUIRE(m == 0 || (rp && agg && prp && (nnz == 0 || (ci && v && conn))));
    return lal::sa_prolongator_fill(c, m, nnz, rp, ci, v, conn, agg, relax, prp, pci, pv);
}
