// SA-AMG hierarchy on the device, the V-cycle preconditioner, SA-AMG-PCG
// and mixed-precision iterative refinement.
//
//   setup      iterative_solvers/amg/saamg.cpp:210-282 (level loop: strength,
//              PMIS, smoothed P, R = P^T, A_c = R (A P); eps halves per level;
//              stop when P has no columns or at min(max_levels, 20) levels)
//   V-cycle    iterative_solvers/amg/amg.cpp:144-267 with apply_smoother(jacobi)
//   PCG        iterative_solvers/krylov/cg.cpp:136-223, convergence test of
//              iterative_solvers/iter_control.cpp:38-91
//
// Everything stays on the device.  Solver scalars (gamma, alpha, beta) are
// formed on the device from per-block partials, so a PCG iteration hands one
// 8-byte residual norm to the host for the convergence test and nothing else.
#include "lal_hier.h"
#include "lal_rowvec.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

namespace lal
{
    int sa_strength(lal_context* c, int m, int nnz, const int* rp, const int* ci,
                    const double* v, double eps, int* conn, arena* a);
    int pmis_aggregate(lal_context* c, int m, int nnz, const int* rp, const int* ci,
                       const int* conn, int64_t* agg, arena* a);
    int sa_prolongator_nnz(lal_context* c, int m, int nnz, const int* rp, const int* ci,
                           const int* conn, const int64_t* agg, int* prp, int* nnz_P, int* n_c,
                           arena* a);
    int sa_prolongator_fill(lal_context* c, int m, int nnz, const int* rp, const int* ci,
                            const double* v, const int* conn, const int64_t* agg, double relax,
                            const int* prp, int* pci, double* pv);
    bool small_fits(int m, long nnz);
    int  small_build(lal_context* c, int m, int nnz, const int* rp, const int* ci,
                     const double* v, double eps, double relax, bool unsmoothed, int* prp,
                     int* pci, double* pv, int* rrp, int* rci, double* rv, int* nnz_P, int* n_c,
                     arena* a);
    int ua_prolongator_nnz(lal_context* c, int m, const int64_t* agg, int* prp, int* nnz_P,
                           int* n_c, arena* a);
    int ua_prolongator_fill(lal_context* c, int m, const int64_t* agg, const int* prp, int* pci,
                            double* pv);
    int transpose_f64(lal_context* c, int m, int n, int nnz, const int* rp, const int* ci,
                      const double* v, int* trp, int* tci, double* tv, arena* a);
    // nnz_a: A's nonzeros, which pick the lanes per row of the product count
    int product(lal_context* c, int m, int k, int n, int nnz_a, const int* arp, const int* aci,
                const double* av, int nnz_b, const int* brp, const int* bci, const double* bv,
                int** crp, int** cci, double** cv, int* nnz_c, arena* mem, arena* work);
}

using lal::converges;
using lal::post_norm;
using lal::wait_scalar;
using lal::csr_dev;
using lal::level_t;
using lal::work;

namespace
{
    template <typename T>
    const T* vals(const csr_dev& A);
    template <>
    const double* vals<double>(const csr_dev& A)
    {
        return A.v;
    }
    template <>
    const float* vals<float>(const csr_dev& A)
    {
        return A.v32;
    }

    // r = b - A x in the level's precision
    template <typename T>
    int residual_t(lal_context* c, const csr_dev& A, const T* Av, const T* x, const T* b, T* r)
    {
        if(sizeof(T) == 8)
            return lal::residual_f64(c, A.d, A.m, A.n, A.nnz, A.rp, A.ci, (const double*)Av,
                                     (const double*)x, (const double*)b, (double*)r);
        return lal::residual_f32(c, A.d, A.m, A.n, A.nnz, A.rp, A.ci, (const float*)Av,
                                 (const float*)x, (const float*)b, (float*)r);
    }

    // Dense inverse of the coarsest operator through its Cholesky factor
    // (FP64, on the host; the operator is small).  Returns false if a pivot
    // is not positive.
    bool dense_inverse(int n, const std::vector<int>& rp, const std::vector<int>& ci,
                       const std::vector<double>& v, std::vector<double>& inv)
    {
        std::vector<double> Lf((size_t)n * n, 0.0);
        for(int i = 0; i < n; i++)
            for(int j = rp[i]; j < rp[i + 1]; j++)
                Lf[(size_t)i * n + ci[j]] = v[j];
        for(int j = 0; j < n; j++)
        {
            double s = Lf[(size_t)j * n + j];
            for(int k = 0; k < j; k++)
                s -= Lf[(size_t)j * n + k] * Lf[(size_t)j * n + k];
            if(!(s > 0.0))
                return false;
            double d             = std::sqrt(s);
            Lf[(size_t)j * n + j] = d;
            for(int i = j + 1; i < n; i++)
            {
                double t = Lf[(size_t)i * n + j];
                for(int k = 0; k < j; k++)
                    t -= Lf[(size_t)i * n + k] * Lf[(size_t)j * n + k];
                Lf[(size_t)i * n + j] = t / d;
            }
        }
        inv.assign((size_t)n * n, 0.0);
        std::vector<double> col(n);
        for(int e = 0; e < n; e++)
        {
            for(int i = 0; i < n; i++)
            {
                double t = (i == e) ? 1.0 : 0.0;
                for(int k = 0; k < i; k++)
                    t -= Lf[(size_t)i * n + k] * col[k];
                col[i] = t / Lf[(size_t)i * n + i];
            }
            for(int i = n - 1; i >= 0; i--)
            {
                double t = col[i];
                for(int k = i + 1; k < n; k++)
                    t -= Lf[(size_t)k * n + i] * col[k];
                col[i] = t / Lf[(size_t)i * n + i];
            }
            for(int i = 0; i < n; i++)
                inv[(size_t)i * n + e] = col[i];
        }
        return true;
    }

    // The dense operator of the V-cycle's small end: the first level from
    // `levels` - 1 down to 1 that is still within lal::CYCLE_ROWS rows, on the
    // fast path with a direct coarsest solve.
    int cycle_operator(lal_hierarchy_t* h, lal::arena* tmp)
    {
        lal_context* c     = h->c;
        int          first = h->levels;
        while(first > 1 && h->L[first - 1].A.m <= lal::CYCLE_ROWS)
            first--;
        const level_t& last = h->L[h->levels];
        if(h->opts.exact || h->lean || h->coarse_kind == 1 || first == h->levels ||
           last.A.m > lal::CYCLE_ROWS)
            return LAL_OK;
        const double* Mc  = h->coarse_kind == 2 ? h->coarse_inv : nullptr;
        int           ldc = last.A.m;
        for(int l = h->levels - 1; l >= first; l--)
        {
            const level_t&   L  = h->L[l];
            const size_t     ld = lal::cycle_ld(L.A.m);
            lal::cycle_level in{L.A.m, L.R.m, L.A.rp, L.A.ci, L.A.v, L.w64.dinv, L.R.rp, L.R.ci,
                                L.R.v, L.Q.rp, L.Q.ci, L.Q.v};
            double *         S = nullptr, *U = nullptr, *M = nullptr;
            LAL_TRY(tmp->get(&S, ld * L.R.m));
            LAL_TRY(tmp->get(&U, ld * L.R.m));
            LAL_TRY((l == first ? &h->mem : tmp)->get(&M, ld * L.A.m));
            LAL_TRY(lal::cycle_matrix(c, in, Mc, ldc, last.A.v, S, U, M));
            Mc  = M;
            ldc = (int)ld;
        }
        h->cycle_first = first;
        h->cycle_op    = const_cast<double*>(Mc);
        return LAL_OK;
    }

    // PCG forms its next direction p = z + beta p inside the product that needs it,
    // for every gathered entry, and spares the pass between (128^2 Poisson 4.2 + 3.8
    // us -> 6.4), where that pays: a second gathered vector costs more the more
    // entries there are, and the more of them a row's neighbours do not share.
    // Whole FP64 and reliable solves, seven pairs in turn, gain of forming it so:
    //   grids, 5 to 7 per row, 8,000 to 65,000 rows 1.05 .. 1.17, 130,000 1.05 .. 1.18,
    //     262,144 (64^3, 512^2) 1.03 .. 1.12, 327,680 1.02 .. 1.04
    //   graphs, 6 to 13 per row, up to 131,072 rows 1.02 .. 1.07; 262,144 rows (1.5 to
    //     3.3 million entries) 1.02 .. 1.04, 0.98, 1.02, 0.96 .. 1.00
    //   graphs, 15 per row, up to 48,000 rows (706,000 entries) 1.01 .. 1.08, 65,536 rows
    //     0.99 .. 1.00, 131,072 0.97 .. 1.03, 250,000 0.93 .. 0.99
    // (pairs of one case differ by 1 to 4 %)
    bool step_pays(const csr_dev& A)
    {
        return A.nnz <= (A.nnz <= 13L * A.m ? 2 << 20 : 706000);
    }

    // A fresh descriptor for an m x n operator of a hierarchy.
    lal_csrmv_info* descr(csr_dev& A, int m, int nnz, int n, int exact)
    {
        A.d         = new lal_csrmv_info;
        A.d->m      = m;
        A.d->nnz    = nnz;
        A.d->exact  = exact;
        A.d->by_nnz = m != n;
        return A.d;
    }

    // Which operators are read with cache-allocating loads, per precision of the
    // cycle: they share lal::CACHE_KEEP_BYTES of the Infinity Cache.  The finest
    // one comes first (a PCG iteration reads it three times), then, beside eight
    // of the iteration's vectors, whole levels from the coarsest up.  Gradient on
    // 64^3, where everything fits: 14.1 ms with the finest alone, 13.25 with all;
    // PCG on 101^3 (FP64), where levels 3 and up fit: 8.65 and 8.54 ms, but 9.03
    // with level 2 and 9.05 with all, since what overflows evicts the rest.
    void choose_kept(lal_hierarchy_t* h)
    {
        for(const size_t prec : {sizeof(double), sizeof(float)})
        {
            const int bit  = prec == sizeof(double) ? 1 : 2;
            size_t    room = lal::CACHE_KEEP_BYTES;
            auto      size = [&](const csr_dev& M) {
                // (a column list adds about a third of an entry per nonzero)
                return !M.d ? 0
                            : (size_t)M.nnz * (prec + (M.d->list_max ? 3 : M.d->d_c16 ? 2 : 4));
            };
            auto take = [&](std::initializer_list<csr_dev*> ops) {
                size_t all = 0;
                for(const csr_dev* M : ops)
                    all += size(*M);
                if(all > room)
                    return false;
                room -= all;
                for(csr_dev* M : ops)
                    if(M->d)
                        M->d->keep |= bit;
                return true;
            };
            if(!take({&h->L[0].A}))
                continue;
            room -= std::min(room, 8 * prec * (size_t)h->L[0].A.m);
            int l = h->levels;
            while(l > 0 && take({&h->L[l].A, &h->L[l - 1].R, &h->L[l - 1].Q}))
                l--;
        }
    }

    int finish_setup(lal_hierarchy_t* h, lal::arena* tmp)
    {
        lal_context* c     = h->c;
        const int    exact = h->opts.exact;
        // level 0 carries the descriptor of the input's validation (the same
        // pattern, copied); the rest are this setup's products.  The fast path
        // reads the operators with 16-bit columns (offsets from each row
        // block's smallest column) where the blocks allow it: 2 bytes per
        // nonzero less, same results.
        std::vector<lal::rb_request> req;
        for(int l = 0; l <= h->levels; l++)
            for(csr_dev* A : {&h->L[l].A, &h->L[l].P, &h->L[l].R, &h->L[l].Q})
                if(A->d == nullptr && (A == &h->L[l].A || (l < h->levels && A->rp)))
                    req.push_back({descr(*A, A->m, A->nnz, A->n, exact), A->rp, A->ci, A->m,
                                   A->nnz, exact == 0, -1, !h->lean && A != &h->L[l].P});
        LAL_TRY(lal::analyse(c, req, &h->mem, tmp));
        if(!exact)
            choose_kept(h);
        lal::f32_copies copies;
        for(int l = 0; l <= h->levels; l++)
        {
            level_t& L = h->L[l];
            LAL_TRY(h->mem.get(&L.w64.x, L.A.m));
            LAL_TRY(h->mem.get(&L.w64.t, L.A.m));
            LAL_TRY(h->mem.get(&L.w64.b, L.A.m));
            LAL_TRY(h->mem.get(&L.w64.r, L.A.m));
            LAL_TRY(h->mem.get(&L.w64.diag, L.A.m));
            LAL_TRY(h->mem.get(&L.w64.dinv, L.A.m));
            const bool       up = l < h->levels, f32 = h->opts.build_f32, q = up && L.Q.rp;
            lal::ready_level r{L.A.m, L.A.rp, L.A.ci, L.A.v, L.w64.diag, L.w64.dinv};
            if(f32)
            {
                LAL_TRY(h->mem.get(&L.A.v32, L.A.nnz));
                for(csr_dev* M : {&L.P, &L.R})
                    if(up)
                    {
                        LAL_TRY(h->mem.get(&M->v32, M->nnz));
                        copies.add(M->v, M->v32, M->nnz);
                    }
                LAL_TRY(h->mem.get(&L.w32.x, L.A.m));
                LAL_TRY(h->mem.get(&L.w32.t, L.A.m));
                LAL_TRY(h->mem.get(&L.w32.b, L.A.m));
                LAL_TRY(h->mem.get(&L.w32.r, L.A.m));
                LAL_TRY(h->mem.get(&L.w32.diag, L.A.m));
                LAL_TRY(h->mem.get(&L.w32.dinv, L.A.m));
                r.v32    = L.A.v32;
                r.d32    = L.w32.diag;
                r.dinv32 = L.w32.dinv;
                if(q)
                    LAL_TRY(h->mem.get(&L.Q.v32, L.Q.nnz));
            }
            if(q)
            {
                r.qrp  = L.Q.rp;
                r.qci  = L.Q.ci;
                r.qv   = L.Q.v;
                r.qv32 = L.Q.v32;
                r.prp  = L.P.rp;
                r.pci  = L.P.ci;
                r.pv   = L.P.v;
            }
            LAL_TRY(lal::make_ready(c, r, q ? std::max(L.A.nnz, L.Q.nnz) : L.A.nnz));
        }
        LAL_TRY(lal::copy_f32(c, copies));
        // coarsest level
        csr_dev& Ac = h->L[h->levels].A;
        if(Ac.m == 1)
        {
            if(Ac.nnz < 1)
            {
                lal::set_last_error("coarsest 1x1 operator has no entry");
                return LAL_ERR_UNSUPPORTED;
            }
            h->coarse_kind = 0;
        }
        else if(h->opts.coarse_solver == 1 && Ac.m <= 4096)
        {
            std::vector<int>    rp(Ac.m + 1), ci(Ac.nnz);
            std::vector<double> v(Ac.nnz), inv;
            LAL_HIP(hipMemcpyAsync(rp.data(), Ac.rp, sizeof(int) * (Ac.m + 1),
                                   hipMemcpyDeviceToHost, c->stream));
            if(Ac.nnz)
            {
                LAL_HIP(hipMemcpyAsync(ci.data(), Ac.ci, sizeof(int) * Ac.nnz,
                                       hipMemcpyDeviceToHost, c->stream));
                LAL_HIP(hipMemcpyAsync(v.data(), Ac.v, sizeof(double) * Ac.nnz,
                                       hipMemcpyDeviceToHost, c->stream));
            }
            LAL_HIP(hipStreamSynchronize(c->stream));
            if(dense_inverse(Ac.m, rp, ci, v, inv))
            {
                LAL_TRY(h->mem.get(&h->coarse_inv, inv.size()));
                LAL_HIP(hipMemcpyAsync(h->coarse_inv, inv.data(), sizeof(double) * inv.size(),
                                       hipMemcpyHostToDevice, c->stream));
                LAL_HIP(hipStreamSynchronize(c->stream));
                h->coarse_kind = 2;
            }
            else
                h->coarse_kind = 1;
        }
        else
            h->coarse_kind = 1;

        LAL_TRY(cycle_operator(h, tmp));

        const int n = h->L[0].A.m;
        LAL_TRY(h->mem.get(&h->res, n));
        LAL_TRY(h->mem.get(&h->z, n));
        LAL_TRY(h->mem.get(&h->p, n));
        LAL_TRY(h->mem.get(&h->q, n));
        LAL_TRY(h->mem.get(&h->s, lal::LAL_SOLVER_SLOTS));
        if(step_pays(h->L[0].A))
            LAL_TRY(h->mem.get(&h->p2, n));
        LAL_TRY(h->mem.get(&h->part_pq, lal::PCG_PARTS));
        LAL_TRY(h->mem.get(&h->part_g, lal::PCG_PARTS));
        LAL_TRY(h->mem.get(&h->part_r, lal::PCG_BLOCKS));
        LAL_TRY(h->mem.get(&h->d_count, 1));
        LAL_TRY(lal_fill_i32(c, (int*)h->d_count, 1, 0));
        if(c->pool->take_note((void**)&h->h_note, (void**)&h->d_note))
            h->pool = c->pool;
        else
        {
            LAL_HIP(hipHostMalloc((void**)&h->h_note, 64,
                                  hipHostMallocMapped | hipHostMallocCoherent));
            std::memset(h->h_note, 0, 64);
            LAL_HIP(hipHostGetDevicePointer((void**)&h->d_note, h->h_note, 0));
        }
        h->h_seq = reinterpret_cast<unsigned*>(h->h_note + 1);
        h->d_seq = reinterpret_cast<unsigned*>(h->d_note + 1);
        if(h->opts.build_f32)
        {
            LAL_TRY(h->mem.get(&h->res32, n));
            LAL_TRY(h->mem.get(&h->z32, n));
            LAL_TRY(h->mem.get(&h->p32, n));
            if(step_pays(h->L[0].A))
                LAL_TRY(h->mem.get(&h->p2_32, n));
            LAL_TRY(h->mem.get(&h->q32, n));
            LAL_TRY(h->mem.get(&h->d32, n));
            h->has32 = true;
        }
        LAL_HIP(hipStreamSynchronize(c->stream));
        return LAL_OK;
    }

    // Level loop of saamg_setup (saamg.cpp:210-282) or, with unsmoothed set,
    // uaamg_setup (uaamg.cpp:125-224): the same strength, PMIS and Galerkin
    // steps around a different prolongator.
    int setup(lal_context* c, int m, int n, int nnz, const int* rp, const int* ci,
              const double* v, const lal_saamg_options& o, lal_hierarchy_t* h,
              bool unsmoothed = false)
    {
        h->c    = c;
        h->opts = o;
        csr_dev& A0 = h->L[0].A;
        A0.m = m;
        A0.n = n;
        A0.nnz = nnz;
        // a level's temporary arrays; a lean build gives them back as soon as they
        // are done with, and lets every step free its own
        std::unique_ptr<lal::arena> tmp;
        auto fresh = [&]() -> int {
            if(tmp && !h->lean)
            {
                tmp->release(lal::arena::mark_t{});
                return LAL_OK;
            }
            if(tmp)
                LAL_HIP(hipStreamSynchronize(c->stream));
            tmp.reset(new lal::arena);
            if(h->lean)
                tmp->tight();
            else
            {
                tmp->use(c->pool);
                tmp->reserve((size_t)nnz * 30 + (size_t)m * 60);
            }
            return LAL_OK;
        };
        LAL_TRY(fresh());
        lal::arena* const work = h->lean ? nullptr : tmp.get();
        LAL_TRY(h->mem.get(&A0.rp, m + 1));
        LAL_TRY(h->mem.get(&A0.ci, nnz));
        LAL_TRY(h->mem.get(&A0.v, nnz));
        LAL_HIP(hipMemcpyAsync(A0.rp, rp, sizeof(int) * (m + 1), hipMemcpyDeviceToDevice,
                               c->stream));
        if(nnz)
        {
            LAL_HIP(hipMemcpyAsync(A0.ci, ci, sizeof(int) * nnz, hipMemcpyDeviceToDevice,
                                   c->stream));
            LAL_HIP(hipMemcpyAsync(A0.v, v, sizeof(double) * nnz, hipMemcpyDeviceToDevice,
                                   c->stream));
        }
        int    max_level = std::min(o.max_levels, 20);
        double eps       = o.eps;
        int    level     = 0;
        while(level < max_level)
        {
            csr_dev& Af = h->L[level].A;
            csr_dev& P  = h->L[level].P;
            csr_dev& R  = h->L[level].R;
            csr_dev& Ac = h->L[level + 1].A;
            LAL_TRY(fresh());
            LAL_TRY(h->mem.get(&P.rp, Af.m + 1));
            int nnzP = 0, nc = 0;
            if(lal::small_fits(Af.m, Af.nnz))
            {
                const int room = std::max(Af.m, Af.nnz);
                LAL_TRY(h->mem.get(&P.ci, room));
                LAL_TRY(h->mem.get(&P.v, room));
                LAL_TRY(h->mem.get(&R.rp, Af.m + 1));
                LAL_TRY(h->mem.get(&R.ci, room));
                LAL_TRY(h->mem.get(&R.v, room));
                LAL_TRY(lal::small_build(c, Af.m, Af.nnz, Af.rp, Af.ci, Af.v, eps, o.relax,
                                         unsmoothed, P.rp, P.ci, P.v, R.rp, R.ci, R.v, &nnzP, &nc,
                                         work));
            }
            else
            {
                int*     conn = nullptr;
                int64_t* agg  = nullptr;
                LAL_TRY(tmp->get(&conn, Af.nnz));
                LAL_TRY(tmp->get(&agg, Af.m));
                LAL_TRY(lal::sa_strength(c, Af.m, Af.nnz, Af.rp, Af.ci, Af.v, eps, conn, work));
                LAL_TRY(lal::pmis_aggregate(c, Af.m, Af.nnz, Af.rp, Af.ci, conn, agg, work));
                if(unsmoothed)
                    LAL_TRY(lal::ua_prolongator_nnz(c, Af.m, agg, P.rp, &nnzP, &nc, work));
                else
                    LAL_TRY(lal::sa_prolongator_nnz(c, Af.m, Af.nnz, Af.rp, Af.ci, conn, agg,
                                                    P.rp, &nnzP, &nc, work));
                if(nc > 0)
                {
                    LAL_TRY(h->mem.get(&P.ci, nnzP));
                    LAL_TRY(h->mem.get(&P.v, nnzP));
                    if(unsmoothed)
                        LAL_TRY(lal::ua_prolongator_fill(c, Af.m, agg, P.rp, P.ci, P.v));
                    else
                        LAL_TRY(lal::sa_prolongator_fill(c, Af.m, Af.nnz, Af.rp, Af.ci, Af.v, conn,
                                                         agg, o.relax, P.rp, P.ci, P.v));
                    // R = P^T
                    LAL_TRY(h->mem.get(&R.rp, nc + 1));
                    LAL_TRY(h->mem.get(&R.ci, nnzP));
                    LAL_TRY(h->mem.get(&R.v, nnzP));
                    LAL_TRY(lal::transpose_f64(c, Af.m, nc, nnzP, P.rp, P.ci, P.v, R.rp, R.ci, R.v,
                                               work));
                }
            }
            if(nc == 0)
            {
                P = csr_dev{};
                R = csr_dev{};
                break;
            }
            P.m   = Af.m;
            P.n   = nc;
            P.nnz = nnzP;
            R.m   = nc;
            R.n   = Af.m;
            R.nnz = nnzP;
            if(h->lean)
                LAL_TRY(fresh());
            // AP = A P (the fast path makes Q of it)
            csr_dev  ap_tmp;
            csr_dev& AP = o.exact || h->lean ? ap_tmp : h->L[level].Q;
            AP.m        = Af.m;
            AP.n        = nc;
            LAL_TRY(lal::product(c, Af.m, Af.n, nc, Af.nnz, Af.rp, Af.ci, Af.v, P.nnz, P.rp,
                                 P.ci, P.v, &AP.rp, &AP.ci, &AP.v, &AP.nnz,
                                 &AP == &ap_tmp ? tmp.get() : &h->mem, work));
            // A_c = R (A P)
            Ac.m = nc;
            Ac.n = nc;
            LAL_TRY(lal::product(c, nc, Af.m, nc, R.nnz, R.rp, R.ci, R.v, AP.nnz, AP.rp, AP.ci,
                                 AP.v, &Ac.rp, &Ac.ci, &Ac.v, &Ac.nnz, &h->mem, work));
            level++;
            eps *= 0.5;
        }
        h->levels = level;
        if(h->lean)
            LAL_TRY(fresh());
        const int st = finish_setup(h, tmp.get());
        (void)hipStreamSynchronize(c->stream); // before the arrays go
        return st;
    }

    // What level 0's kernels do for the solver besides the cycle (merged()
    // holds): the residual pass finishes the reduction `post`, the correction
    // leaves <dot.w, z>'s partials in dot.part.
    struct cycle_extra
    {
        lal::post_args post{};
        lal::row_extra dot{};
    };

    // One pre-sweep and a post-sweep on the fast path: the residual pass also
    // leaves y = x + r / a_ii, and the way up is y + Q e.
    bool merged(const lal_hierarchy_t* h, int l, int n1, int n2)
    {
        return !h->opts.exact && n1 == 1 && n2 >= 1 && l < h->levels && h->L[l].Q.rp;
    }

    // One V-cycle at level l for rhs b with the initial guess zero.  The
    // result lands in dst when given, else in a level buffer; *out gets it.
    template <typename T>
    int vcycle(lal_hierarchy_t* h, int l, const T* b, T* dst, int n1, int n2, bool xinit,
               T** out, const cycle_extra& ex = {})
    {
        lal_context* c = h->c;
        level_t&     L = h->L[l];
        work<T>&     W = h->w<T>(l);
        const csr_dev& A = L.A;
        const T*       Av = vals<T>(A);
        // Fast path with one pre-sweep: the sweep from zero is x = b/a_ii,
        // written by whoever produced b (the restriction above, or the PCG
        // update for level 0) when xinit is set; this level then only forms
        // r = b - A x.
        const bool fast = !h->opts.exact && n1 == 1;
        if(fast && n2 == 1 && l == h->cycle_first)
        {
            T* res = dst ? dst : W.t;
            LAL_TRY(lal::cycle_apply<T>(c, A.m, h->cycle_op, b, res));
            *out = res;
            return LAL_OK;
        }
        if(l == h->levels)
        {
            T* x = dst ? dst : W.x;
            if(h->coarse_kind == 0)
                LAL_TRY(lal::coarse_scalar<T>(c, Av, b, x));
            else if(h->coarse_kind == 2)
                LAL_TRY(lal::coarse_dense<T>(c, A.m, h->coarse_inv, b, x));
            else
                LAL_TRY(lal::coarse_gs<T>(c, A.m, A.rp, A.ci, Av, b, x));
            *out = x;
            return LAL_OK;
        }
        T* cur   = W.x;
        T* other = W.t;
        const bool post_merged = merged(h, l, n1, n2); // y lies in W.t
        if(n1 == 0)
        {
            // x = 0 and r = b - A*0, which is b bit for bit
            LAL_HIP(hipMemsetAsync(cur, 0, sizeof(T) * A.m, c->stream));
            LAL_HIP(hipMemcpyAsync(W.r, b, sizeof(T) * A.m, hipMemcpyDeviceToDevice, c->stream));
        }
        else if(fast)
        {
            if(!xinit)
                LAL_TRY(lal::mul_elem<T>(c, A.m, b, W.dinv, cur));
            if(post_merged)
                LAL_TRY(lal::residual_smoothed<T>(c, A.d, A.m, A.rp, A.ci, Av, cur, W.dinv, b, W.r,
                                                  other, ex.post));
            else
                LAL_TRY(residual_t<T>(c, A, Av, cur, b, W.r));
        }
        else
        {
            LAL_TRY(lal::jacobi0_residual<T>(c, A.d, A.m, A.rp, A.ci, Av, W.diag, W.dinv, b, cur,
                                             W.r));
            if(n1 > 1)
            {
                for(int k = 1; k < n1; k++)
                {
                    LAL_TRY(lal::jacobi_sweep<T>(c, A.d, A.m, A.rp, A.ci, Av, W.diag, W.dinv,
                                                 cur, b, other));
                    std::swap(cur, other);
                }
                LAL_TRY(residual_t<T>(c, A, Av, cur, b, W.r));
            }
        }
        // restriction: b_{l+1} = R r (and, on the fast path, x_{l+1} = b_{l+1}/a_ii)
        const csr_dev& R  = L.R;
        work<T>&       Wc = h->w<T>(l + 1);
        if(fast)
            LAL_TRY(lal::restrict_init<T>(c, R.d, R.m, R.rp, R.ci, vals<T>(R), W.r, Wc.dinv,
                                          Wc.b, Wc.x));
        else
            LAL_TRY(lal::csrmv(c, R.d, R.m, R.n, R.nnz, 1.0, R.rp, R.ci, vals<T>(R), W.r, 0.0,
                               Wc.b));
        T* ec = nullptr;
        LAL_TRY(vcycle<T>(h, l + 1, Wc.b, nullptr, n1, n2, fast, &ec));
        int done = 0; // post-sweeps behind us
        if(post_merged)
        {
            // other = y; the result may go straight to dst
            T* o = n2 == 1 && dst ? dst : cur;
            LAL_TRY(lal::add_product<T>(c, L.Q.d, L.Q.m, L.Q.rp, L.Q.ci, vals<T>(L.Q), ec, other,
                                        o, ex.dot));
            cur  = o;
            done = 1;
        }
        else
        {
            // prolongation and correction: x += P ec
            const csr_dev& P = L.P;
            LAL_TRY(lal::csrmv(c, P.d, P.m, P.n, P.nnz, 1.0, P.rp, P.ci, vals<T>(P), ec, 1.0,
                               cur));
        }
        for(int k = done; k < n2; k++)
        {
            T* o = (k == n2 - 1 && dst) ? dst : other;
            LAL_TRY(lal::jacobi_sweep<T>(c, A.d, A.m, A.rp, A.ci, Av, W.diag, W.dinv, cur, b,
                                         o));
            other = cur;
            cur   = o;
        }
        if(dst && cur != dst)
        {
            LAL_HIP(hipMemcpyAsync(dst, cur, sizeof(T) * A.m, hipMemcpyDeviceToDevice,
                                   c->stream));
            cur = dst;
        }
        *out = cur;
        return LAL_OK;
    }

    template <typename T>
    int precond(lal_hierarchy_t* h, const T* r, T* z, int n1, int n2, bool xinit = false,
                const cycle_extra& ex = {})
    {
        T* out = nullptr;
        return vcycle<T>(h, 0, r, z, n1, n2, xinit, &out, ex);
    }

    // precond() for the solvers' own vectors (r, z fixed per hierarchy and
    // precision): with at least one pre-sweep the V-cycle is kernels and
    // device copies only.  On a small finest level (at most GRAPH_MAX_ROWS
    // rows), where every kernel is short and the host's launches bound the cycle,
    // it is captured as a HIP graph on its second use and replayed after
    // (lal::captured): PCG on 2D Poisson 128^2, 16,384 rows, 1.37 ms against 1.51
    // to 1.56 launched eagerly by a busy host.  The host launches at one of two
    // speeds, by process; a graph takes the same time in both.  Whole solves,
    // graph / eager fast / eager slow (us): 2D 66,049 rows 2050 / 1970 / 2210 to
    // 2460, 131,044 rows 2270 to 2360 / 2120 to 2160 / 2430 to 2620, 261,632 rows
    // 2770 to 2920 / 2560 to 2750 / 2840 to 3010; 3D diffusion 91,125 rows 1510 /
    // 1390 to 1440 / 1550 to 1690, 166,375 rows 1790 / 1670 to 1690 / 1810 to 1900,
    // 262,144 rows 1980 to 2070 / 1870 to 1980 / 2000 to 2060 (gradient on 64^3:
    // 11.9 and 12.4 against 11.3 and 11.8 ms).  The line is where what the slow
    // speed loses no longer outweighs what the fast one gains.
    constexpr int GRAPH_MAX_ROWS = 131072;

    template <typename T>
    int precond_graphed(lal_hierarchy_t* h, const T* r, T* z, int n1, int n2,
                        bool xinit = false, const cycle_extra& ex = {})
    {
        if(n1 < 1 || h->L[0].A.m > GRAPH_MAX_ROWS)
            return precond<T>(h, r, z, n1, n2, xinit, ex);
        // (ex is the same for every call with these flags: the solvers' own
        // buffers; the inner product's other vector goes with the precision)
        const int kind = lal::KIND_PRECOND + (sizeof(T) == 4 ? 1 : 0) + 2 * (int)xinit +
                         (ex.post.part ? 4 : 0) + (ex.dot.part ? 8 : 0) + (ex.dot.wide ? 16 : 0);
        return lal::captured(h, z, r, n1, n2, 0, 0, kind,
                             [&] { return precond<T>(h, r, z, n1, n2, xinit, ex); });
    }

    // z = one V-cycle on r, and the partials of <z, w> (w: the residual in the
    // solver's precision) in h->part_g, *n_g of them.  seq given: the norm
    // max|r| in h->part_r (n_r partials) is handed to the host on the way.
    // Where the cycle's own kernels can do either, no launch of its own is spent.
    template <typename T, typename W>
    int apply_dot(lal_hierarchy_t* h, const T* r, T* z, const W* w, int n1, int n2, bool xinit,
                  int n_r, unsigned* seq, int* n_g)
    {
        const csr_dev& Q    = h->L[0].Q;
        const bool     fold = merged(h, 0, n1, n2);
        cycle_extra    ex;
        if(seq)
            LAL_TRY(post_norm(h, n_r, lal::S_RNORM, seq, fold ? &ex.post : nullptr));
        if(fold && n2 == 1 && lal::can_add_dot<T>(Q.d, Q.m, Q.rp, Q.ci, vals<T>(Q)))
        {
            ex.dot.part = h->part_g;
            ex.dot.w    = w;
            ex.dot.wide = sizeof(W) > sizeof(T);
        }
        LAL_TRY(precond_graphed<T>(h, r, z, n1, n2, xinit, ex));
        *n_g = ex.dot.part ? Q.d->nblocks : lal::PCG_BLOCKS;
        return ex.dot.part ? LAL_OK
                           : lal::dot_partials<T, W>(h->c, h->L[0].A.m, z, w, h->part_g);
    }

    // q = A p for the next step, with the partials of <q, p>.  stale: p is still the
    // last direction, and p = z + beta p comes first (beta from the partials of
    // <z, r> and its last value; s[S_GAMMA + cur] gets the new one), inside the
    // product where it takes that, which leaves the direction in *p_other.
    template <typename T>
    int next_product(lal_hierarchy_t* h, const csr_dev& A, const T* Av, const T* z, bool stale,
                     T** p, T** p_other, T* q, int n_g, int cur, int* n_pq)
    {
        lal_context* c    = h->c;
        double*      prev = h->s + lal::S_GAMMA + (cur ^ 1);
        double*      now  = h->s + lal::S_GAMMA + cur;
        bool         done = false;
        if(stale && *p_other != nullptr && step_pays(A))
            LAL_TRY(lal::step_dot<T>(c, A.d, A.m, A.n, A.rp, A.ci, Av, z, *p, *p_other, q,
                                     h->part_g, n_g, prev, now, h->part_pq, n_pq, &done));
        if(done)
        {
            std::swap(*p, *p_other);
            return LAL_OK;
        }
        if(stale)
            LAL_TRY(lal::update_p<T, T>(c, A.m, z, *p, h->part_g, n_g, prev, now));
        return lal::product_dot<T>(c, A.d, A.m, A.n, A.nnz, A.rp, A.ci, Av, *p, q, h->part_pq,
                                   n_pq);
    }

    // cg_solver::solve_precond on the device.  T = double uses the FP64
    // levels and workspaces, T = float the FP32 ones.  The Krylov products
    // use `op` when given (a caller's matrix of the finest level's size, FP64
    // only), else the matrix the hierarchy was built from.
    template <typename T>
    int pcg(lal_hierarchy_t* h, const T* b, T* x, T* res, T* z, T* p, T* q, double rel_tol,
            double abs_tol, int max_iter, int n1, int n2, lal_solve_info* info,
            const csr_dev* op = nullptr, int smoother = 0)
    {
        lal_context*   c  = h->c;
        const csr_dev& A  = op ? *op : h->L[0].A;
        const int      n  = A.m;
        const T*       Av = vals<T>(A);
        double*        s  = h->s;
        if(sizeof(T) == 8)
            LAL_TRY(lal::residual_f64(c, A.d, n, A.n, A.nnz, A.rp, A.ci, (const double*)Av,
                                      (const double*)x, (const double*)b, (double*)res));
        else
            LAL_TRY(lal::residual_f32(c, A.d, n, A.n, A.nnz, A.rp, A.ci, (const float*)Av,
                                      (const float*)x, (const float*)b, (float*)res));
        unsigned seq       = 0;
        double   init      = 0.0;
        LAL_TRY(lal::norm_partials<T>(c, n, res, h->part_r));
        LAL_TRY(post_norm(h, lal::PCG_BLOCKS, lal::S_RNORM0, &seq));
        LAL_TRY(wait_scalar(h, seq, lal::S_RNORM0, &init));
        // the preconditioner: one V-cycle from zero, with the Jacobi fast path
        // or (smoother != 0, FP64 only) another smoother of the AMG cycles
        int        n_pq = 0, n_g = 0;
        const int  n_r   = lal::update_blocks(n);
        auto       apply = [&](bool xinit, unsigned* norm) -> int {
            if(smoother == 0)
                return apply_dot<T, T>(h, res, z, res, n1, n2, xinit, n_r, norm, &n_g);
            if(norm)
                LAL_TRY(post_norm(h, n_r, lal::S_RNORM, norm));
            LAL_TRY(lal::vcycle_smoothed(h, (const double*)res, (double*)z, n1, n2, smoother));
            n_g = lal::PCG_BLOCKS;
            return lal::dot_partials<T, T>(c, n, z, res, h->part_g);
        };
        LAL_TRY(apply(false, nullptr));
        LAL_HIP(hipMemcpyAsync(p, z, sizeof(T) * n, hipMemcpyDeviceToDevice, c->stream));
        int cur = 0; // generation of s[S_GAMMA]
        LAL_TRY(lal::finish_partials(c, 0, {h->part_g, n_g, s + lal::S_GAMMA}));
        double rn   = init;
        int    iter = 0;
        bool   conv = false;
        double r_prev = init, rate = 0.5; // last norm, observed reduction per step
        T*     p_other = sizeof(T) == 8 ? (T*)h->p2 : (T*)h->p2_32; // (or null)
        bool   stale   = false; // p is still the last direction: z is to be added
        while(!(iter > max_iter))
        {
            LAL_TRY(next_product<T>(h, A, Av, z, stale, &p, &p_other, q, n_g, cur, &n_pq));
            // with one pre-sweep on the fast path, the update also writes the
            // V-cycle's first Jacobi iterate x0 = r / a_ii
            const bool fast = !h->opts.exact && n1 == 1 && h->levels > 0 && smoother == 0;
            work<T>&   W0   = h->w<T>(0);
            LAL_TRY(lal::update_xr<T, T>(c, n, p, q, x, res, h->part_pq, n_pq,
                                         s + lal::S_GAMMA + cur, h->part_r, s + lal::S_ALPHA,
                                         W0.dinv, fast ? W0.x : nullptr, nullptr));
            // The next preconditioner application depends on r only: it is
            // queued before the host looks at the norm, so the GPU does not
            // wait for the convergence test -- unless the observed rate of
            // reduction predicts that this step converges, when the host
            // decides first so that no V-cycle is spent after the last step.
            const bool near = lal::near_tolerance(r_prev, rate, init, rel_tol, abs_tol);
            LAL_TRY(near ? post_norm(h, n_r, lal::S_RNORM, &seq) : apply(fast, &seq));
            LAL_TRY(wait_scalar(h, seq, lal::S_RNORM, &rn));
            lal::observe_rate(rn, &r_prev, &rate);
            if(std::isnan(rn))
                break; // a NaN in the residual: not converged
            if(converges(rn, init, rel_tol, abs_tol))
            {
                conv = true;
                break;
            }
            if(near)
                LAL_TRY(apply(fast, nullptr));
            stale = true;
            cur ^= 1;
            iter++;
        }
        if(info)
        {
            info->iterations       = iter;
            info->converged        = conv;
            info->initial_res_norm = init;
            info->final_res_norm   = rn;
        }
        return LAL_OK;
    }

    // cg_solver::solve_precond with the Krylov vectors (x, r, p, q), the
    // operator product and every inner product in FP64 and the V-cycle on the
    // FP32 levels.  The residual's FP32 copy and the V-cycle's first Jacobi
    // iterate are written by the FP64 update kernel, and <z, r> / p = z + beta p
    // read the FP32 z directly, so the precision change costs no extra pass.
    // The V-cycle input is r scaled by sigma = 2^-k, k the binary exponent of
    // ||r0||_inf, and rounded to FP32, so its entries stay in FP32's range
    // whatever b's magnitude.  PCG is invariant to a constant scaling of the
    // preconditioner (alpha takes 1/sigma, beta is unchanged), and a power of
    // two scales every iterate exactly, so the iterates are those of the
    // unscaled V-cycle.
    int pcg_mixed(lal_hierarchy_t* h, const double* b, double* x, double rel_tol,
                  double abs_tol, int max_iter, int n1, int n2, lal_solve_info* info)
    {
        lal_context*   c   = h->c;
        const csr_dev& A   = h->L[0].A;
        const int      n   = A.m;
        double*        s   = h->s;
        double*        res = h->res;
        double*        p   = h->p;
        double*        q   = h->q;
        float*         r32 = h->res32;
        float*         z32 = h->z32;
        LAL_TRY(lal::residual_f64(c, A.d, n, A.n, A.nnz, A.rp, A.ci, A.v, x, b, res));
        unsigned seq       = 0;
        double   init      = 0.0;
        LAL_TRY(lal::norm_partials<double>(c, n, res, h->part_r));
        LAL_TRY(post_norm(h, lal::PCG_BLOCKS, lal::S_RNORM0, &seq));
        LAL_TRY(wait_scalar(h, seq, lal::S_RNORM0, &init));
        const double sigma = init > 0.0 && std::isfinite(init) ? std::ldexp(1.0, -std::ilogb(init))
                                                               : 1.0;
        LAL_TRY(lal::scale_cast_f64_f32(c, n, res, sigma, r32));
        int       n_pq = 0, n_g = 0;
        const int n_r   = lal::update_blocks(n);
        auto      apply = [&](bool xinit, unsigned* norm) {
            return apply_dot<float, double>(h, r32, z32, res, n1, n2, xinit, n_r, norm, &n_g);
        };
        LAL_TRY(apply(false, nullptr));
        LAL_TRY(lal_convert_f32_f64(c, z32, p, (size_t)n));
        int cur = 0; // generation of s[S_GAMMA]
        LAL_TRY(lal::finish_partials(c, 0, {h->part_g, n_g, s + lal::S_GAMMA}));
        double       rn   = init;
        int          iter = 0;
        bool         conv = false;
        const bool   fast = !h->opts.exact && n1 == 1 && h->levels > 0;
        work<float>& W0   = h->w<float>(0);
        double       r_prev = init, rate = 0.5;
        while(!(iter > max_iter))
        {
            LAL_TRY(lal::product_dot<double>(c, A.d, n, A.n, A.nnz, A.rp, A.ci, A.v, p, q,
                                             h->part_pq, &n_pq));
            LAL_TRY(lal::update_xr<double, float>(c, n, p, q, x, res, h->part_pq, n_pq,
                                                  s + lal::S_GAMMA + cur, h->part_r,
                                                  s + lal::S_ALPHA, W0.dinv,
                                                  fast ? W0.x : nullptr, r32, sigma));
            const bool near = lal::near_tolerance(r_prev, rate, init, rel_tol, abs_tol);
            LAL_TRY(near ? post_norm(h, n_r, lal::S_RNORM, &seq) : apply(fast, &seq));
            LAL_TRY(wait_scalar(h, seq, lal::S_RNORM, &rn));
            lal::observe_rate(rn, &r_prev, &rate);
            if(std::isnan(rn))
                break; // a NaN in the residual: not converged
            if(converges(rn, init, rel_tol, abs_tol))
            {
                conv = true;
                break;
            }
            if(near)
                LAL_TRY(apply(fast, nullptr));
            LAL_TRY(lal::update_p<float, double>(c, n, z32, p, h->part_g, n_g,
                                                 s + lal::S_GAMMA + cur,
                                                 s + lal::S_GAMMA + (cur ^ 1)));
            cur ^= 1;
            iter++;
        }
        if(info)
        {
            info->iterations       = iter;
            info->outer_iterations = 0;
            info->converged        = conv;
            info->initial_res_norm = init;
            info->final_res_norm   = rn;
        }
        return LAL_OK;
    }
}

namespace
{
    // cg_solver::solve_precond (cg.cpp:136-223) with the Krylov recurrences in
    // FP32 and reliable updates (Sleijpen and van der Vorst, 1996) in FP64.
    // The operator product q = A p, the vectors r, p, q, z and the correction
    // y run in FP32 (A's FP32 values, the FP32 V-cycle); inner products
    // accumulate in FP64.  r is the FP64 residual scaled by 1/||r0||, so its
    // entries stay in FP32's normal range whatever b's magnitude.  When the
    // recursive residual has fallen by `delta` since the last update, or meets
    // the tolerance, the FP64 solution takes the correction (x += y ||r0||)
    // and the recursive residual is replaced by the true FP64 residual
    // b - A x; convergence is declared on that true residual only.  The
    // Krylov space is kept across updates, so the iteration count stays that
    // of the FP64 solve while every pass but the updates moves FP32 data;
    // only an update that fails to cut the true residual tenfold restarts it.
    int pcg_reliable(lal_hierarchy_t* h, const double* b, double* x, double rel_tol,
                     double abs_tol, int max_iter, int n1, int n2, double delta,
                     lal_solve_info* info)
    {
        lal_context*   c     = h->c;
        const csr_dev& A     = h->L[0].A;
        const int      n     = A.m;
        const float*   Av32  = vals<float>(A);
        double*        s     = h->s;
        double*        r64   = h->res;
        float*         r32   = h->res32;
        float*         z32   = h->z32;
        float*         p32   = h->p32;
        float*         q32   = h->q32;
        float*         y32   = h->d32;
        unsigned       seq       = 0;
        double         init      = 0.0;
        LAL_TRY(lal::residual_f64(c, A.d, n, A.n, A.nnz, A.rp, A.ci, A.v, x, b, r64));
        LAL_TRY(lal::norm_partials<double>(c, n, r64, h->part_r));
        LAL_TRY(post_norm(h, lal::PCG_BLOCKS, lal::S_RNORM0, &seq));
        LAL_TRY(wait_scalar(h, seq, lal::S_RNORM0, &init));
        double rn   = init; // true or recursive inf-norm, unscaled
        int    iter = 0, updates = 0;
        bool   conv = converges(rn, init, rel_tol, abs_tol);
        if(!conv)
        {
            const double sigma = 1.0 / init;
            LAL_TRY(lal::scale_cast_f64_f32(c, n, r64, sigma, r32));
            LAL_HIP(hipMemsetAsync(y32, 0, sizeof(float) * n, c->stream));
            int       n_pq = 0, n_g = 0;
            const int n_r   = lal::update_blocks(n);
            auto      apply = [&](bool xinit, unsigned* norm) {
                return apply_dot<float, float>(h, r32, z32, r32, n1, n2, xinit, n_r, norm, &n_g);
            };
            LAL_TRY(apply(false, nullptr));
            LAL_HIP(hipMemcpyAsync(p32, z32, sizeof(float) * n, hipMemcpyDeviceToDevice,
                                   c->stream));
            int cur = 0; // generation of s[S_GAMMA]
            LAL_TRY(lal::finish_partials(c, 0, {h->part_g, n_g, s + lal::S_GAMMA}));
            const bool   fast  = !h->opts.exact && n1 == 1 && h->levels > 0;
            work<float>& W0    = h->w<float>(0);
            float*       p_other = h->p2_32;
            bool         stale   = false; // p32 is still the last direction
            double       r_upd  = init; // true residual norm at the last update
            double       r_prev = init, rate = 0.5; // last norm, observed reduction per step
            int          since  = 0, longest = 0; // steps since the last update; between two at most
            while(!(iter > max_iter))
            {
                LAL_TRY(next_product<float>(h, A, Av32, z32, stale, &p32, &p_other, q32, n_g, cur,
                                            &n_pq));
                LAL_TRY(lal::update_xr<float, float>(c, n, p32, q32, y32, r32, h->part_pq, n_pq,
                                                     s + lal::S_GAMMA + cur, h->part_r,
                                                     s + lal::S_ALPHA, W0.dinv,
                                                     fast ? W0.x : nullptr, nullptr));
                // The next V-cycle is queued before the host reads the norm,
                // unless the observed rate of reduction predicts that this step
                // crosses the update threshold: then the host decides first, so
                // that no V-cycle is spent on a residual about to be replaced.
                const double threshold = std::max(std::max(delta * r_upd, rel_tol * init),
                                                  abs_tol);
                const bool   near      = lal::near_threshold(r_prev, rate, threshold);
                LAL_TRY(near ? post_norm(h, n_r, lal::S_RNORM, &seq) : apply(fast, &seq));
                double rs = 0.0;
                LAL_TRY(wait_scalar(h, seq, lal::S_RNORM, &rs));
                rn = rs * init;
                lal::observe_rate(rn, &r_prev, &rate);
                if(std::isnan(rn))
                    break;
                // A recurrence whose kept direction no longer fits its replaced
                // residual can drift above the last update's norm for thousands of
                // steps (face diffusion 96^3, 1e-12: a true residual of 1.6e-12
                // after 360 steps, the next update 1900 later).  One that takes
                // four times as long as any before it is taken for such: the
                // update comes now, and restarts.
                since++;
                const bool lost   = updates > 0 && since > 4 * std::max(longest, 25);
                const bool update = lost || rn <= delta * r_upd ||
                                    converges(rn, init, rel_tol, abs_tol);
                bool       restart = false;
                if(update)
                {
                    // x += ||r0|| y in FP64; r <- the true residual (scaled)
                    LAL_TRY(lal::axpy_f32_f64(c, n, init, y32, x));
                    LAL_HIP(hipMemsetAsync(y32, 0, sizeof(float) * n, c->stream));
                    LAL_TRY(lal::residual_f64(c, A.d, n, A.n, A.nnz, A.rp, A.ci, A.v, x, b,
                                              r64));
                    LAL_TRY(lal::norm_partials<double>(c, n, r64, h->part_r));
                    LAL_TRY(post_norm(h, lal::PCG_BLOCKS, lal::S_RNORM, &seq));
                    LAL_TRY(lal::scale_cast_f64_f32(c, n, r64, sigma, r32));
                    LAL_TRY(wait_scalar(h, seq, lal::S_RNORM, &rn));
                    updates++;
                    // An update that did not cut the true residual tenfold
                    // means the FP32 recurrence has drifted from the FP64 system
                    // (badly conditioned operators): the kept search direction
                    // no longer belongs to the new residual, so the Krylov space
                    // restarts from it (p = z), as iterative refinement would.
                    // Healthy runs (a reduction near delta per update) never
                    // restart and keep their iterates.
                    restart = lost || rn > 0.1 * r_upd;
                    longest = std::max(longest, since);
                    since   = 0;
                    r_upd   = rn;
                    r_prev  = rn;
                    if(std::isnan(rn))
                        break;
                    if(converges(rn, init, rel_tol, abs_tol))
                    {
                        conv = true;
                        break;
                    }
                    LAL_TRY(apply(false, nullptr));
                }
                else if(near)
                    LAL_TRY(apply(fast, nullptr));
                if(restart)
                {
                    LAL_HIP(hipMemcpyAsync(p32, z32, sizeof(float) * n, hipMemcpyDeviceToDevice,
                                           c->stream));
                    LAL_TRY(lal::finish_partials(c, 0,
                                                 {h->part_g, n_g, s + lal::S_GAMMA + (cur ^ 1)}));
                }
                stale = !restart;
                cur ^= 1;
                iter++;
            }
        }
        if(info)
        {
            info->iterations       = iter;
            info->outer_iterations = updates;
            info->converged        = conv;
            info->initial_res_norm = init;
            info->final_res_norm   = rn;
        }
        return LAL_OK;
    }
}

namespace lal
{
    // True when the norm r_prev, reduced once more at the observed rate, is
    // predicted to meet the threshold (or to come within 25 % of it).
    bool near_threshold(double r_prev, double rate, double threshold)
    {
        return r_prev * rate <= 1.25 * threshold;
    }

    bool near_tolerance(double r_prev, double rate, double init, double rel_tol, double abs_tol)
    {
        return near_threshold(r_prev, rate, std::max(rel_tol * init, abs_tol));
    }

    // Records the reduction of the norm over the last step, clamped to
    // [0.05, 1] (a NaN norm gives 0.05).
    void observe_rate(double rn, double* r_prev, double* rate)
    {
        *rate   = std::min(1.0, std::max(0.05, rn / *r_prev));
        *r_prev = rn;
    }

    bool converges(double res, double init, double rel_tol, double abs_tol)
    {
        if(std::isnan(res) || std::isnan(init))
            return false;
        if(res <= abs_tol)
            return true;
        if(res / init <= rel_tol)
            return true;
        return false;
    }

    int post_norm(lal_hierarchy_t* h, int count, int slot, unsigned* seq, post_args* later)
    {
        const post_args a{h->part_r, count, h->s + slot, h->d_note, h->d_seq, h->d_count};
        *seq = ++h->seq;
        if(later == nullptr)
            return finish_partials(h->c, 1, a);
        *later = a;
        return LAL_OK;
    }

    int wait_scalar(lal_hierarchy_t* h, unsigned seq, int slot, double* v)
    {
        bool there = false;
        LAL_TRY(poll_word(h->c, h->h_seq, seq, &there));
        if(there)
            *v = *reinterpret_cast<volatile double*>(h->h_note);
        else // the stream has drained: read the device copy instead
            LAL_HIP(hipMemcpy(v, h->s + slot, sizeof(double), hipMemcpyDeviceToHost));
        return LAL_OK;
    }
}

extern "C" void lal_saamg_default_options(lal_saamg_options* o)
{
    if(!o)
        return;
    o->max_levels    = 20;
    o->eps           = 0.08;
    o->relax         = 2.0 / 3.0;
    o->coarse_solver = 1;
    o->exact         = 0;
    o->build_f32     = 0;
}

extern "C" void lal_solve_default_options(lal_solve_options* o)
{
    if(!o)
        return;
    o->rel_tol        = 1e-6;
    o->abs_tol        = 1e-6;
    o->max_iter       = 1000;
    o->n1             = 1;
    o->n2             = 1;
    o->inner_rel_tol  = 1e-4;
    o->inner_max_iter = 200;
    o->max_outer      = 30;
    o->smoother       = 0;
}

namespace
{
    int setup_entry(lal_handle c, int m, int n, int nnz, const int* rp, const int* ci,
                    const double* v, const lal_saamg_options* opts, lal_hierarchy* out,
                    bool unsmoothed)
    {
        LAL_REQUIRE(c != nullptr && out != nullptr && m >= 1 && n == m && nnz >= 0);
        LAL_REQUIRE(rp != nullptr && (nnz == 0 || (ci && v)));
        *out = nullptr;
        lal_saamg_options o;
        lal_saamg_default_options(&o);
        if(unsmoothed)
            o.eps = 0.001;
        if(opts)
            o = *opts;
        LAL_REQUIRE(o.max_levels >= 0 && o.eps >= 0.0);
        // validate the input pattern before any setup kernel gathers through
        // it; the analysis describes the finest operator (a copy of the same
        // pattern), so the hierarchy keeps it for level 0
        for(const bool lean : {false, true})
        {
            auto* h = new lal_hierarchy_t;
            h->lean = lean;
            // A hierarchy takes about 140 to 175 bytes per nonzero of a 7-point
            // operator with the column lists and the FP32 levels, less without:
            // the first chunk holds most of it (a hipMalloc and hipFree of
            // hundreds of megabytes take 0.3 ms together), and the arena grows by
            // half its size.
            h->mem.use(c->pool);
            if(lean)
                h->mem.tight();
            else
                h->mem.reserve((size_t)nnz * ((o.exact ? 40 : 80) + (o.build_f32 ? 40 : 0)) +
                               (size_t)m * (o.build_f32 ? 200 : 100));
            int s = lal::analyse(c, {{descr(h->L[0].A, m, nnz, n, o.exact), rp, ci, m, nnz,
                                      o.exact == 0, n}}, &h->mem, nullptr);
            if(s == LAL_OK)
                s = setup(c, m, n, nnz, rp, ci, v, o, h, unsmoothed);
            if(s == LAL_OK)
            {
                c->hierarchies.push_back(h);
                *out = h;
                return LAL_OK;
            }
            (void)hipStreamSynchronize(c->stream);
            delete h;
            if(s != LAL_ERR_OOM)
                return s;
        }
        return LAL_ERR_OOM;
    }
}

namespace lal
{
    void detach_hierarchies(lal_context* c)
    {
        for(lal_hierarchy_t* h : c->hierarchies)
            h->c = nullptr;
        c->hierarchies.clear();
    }
}

extern "C" void lal_uaamg_default_options(lal_saamg_options* o)
{
    lal_saamg_default_options(o);
    if(o)
        o->eps = 0.001;
}

extern "C" int lal_uaamg_setup(lal_handle c, int m, int n, int nnz, const int* rp,
                               const int* ci, const double* v, const lal_saamg_options* opts,
                               lal_hierarchy* out)
{
    return setup_entry(c, m, n, nnz, rp, ci, v, opts, out, true);
}

extern "C" int lal_saamg_setup(lal_handle c, int m, int n, int nnz, const int* rp,
                               const int* ci, const double* v, const lal_saamg_options* opts,
                               lal_hierarchy* out)
{
    return setup_entry(c, m, n, nnz, rp, ci, v, opts, out, false);
}

extern "C" int lal_hierarchy_destroy(lal_hierarchy h)
{
    if(h)
    {
        if(h->c)
        {
            (void)hipStreamSynchronize(h->c->stream);
            auto& v = h->c->hierarchies;
            v.erase(std::remove(v.begin(), v.end(), h), v.end());
        }
        else
            (void)hipDeviceSynchronize(); // its context is gone: wait for all work
        delete h;
    }
    return LAL_OK;
}

extern "C" int lal_hierarchy_levels(lal_hierarchy h, int* total)
{
    LAL_REQUIRE(h != nullptr && total != nullptr);
    *total = h->levels;
    return LAL_OK;
}

extern "C" int lal_hierarchy_level(lal_hierarchy h, int level, int kind, int* m, int* n,
                                   int* nnz, const int** rp, const int** ci, const double** v)
{
    LAL_REQUIRE(h != nullptr && m && n && nnz && rp && ci && v);
    LAL_REQUIRE(level >= 0 && kind >= 0 && kind <= 2);
    LAL_REQUIRE(kind == 0 ? level <= h->levels : level < h->levels);
    const csr_dev& A = kind == 0 ? h->L[level].A : (kind == 1 ? h->L[level].P : h->L[level].R);
    *m   = A.m;
    *n   = A.n;
    *nnz = A.nnz;
    *rp  = A.rp;
    *ci  = A.ci;
    *v   = A.v;
    return LAL_OK;
}

extern "C" int lal_hierarchy_column_bytes(lal_hierarchy h, int level, int kind, int* bytes)
{
    LAL_REQUIRE(h != nullptr && bytes != nullptr);
    LAL_REQUIRE(level >= 0 && kind >= 0 && kind <= 2);
    LAL_REQUIRE(kind == 0 ? level <= h->levels : level < h->levels);
    const csr_dev& A = kind == 0 ? h->L[level].A : (kind == 1 ? h->L[level].P : h->L[level].R);
    *bytes           = A.d && A.d->d_c16 ? 2 : 4;
    return LAL_OK;
}

extern "C" int lal_amg_precond_f64(lal_handle c, lal_hierarchy h, const double* r, double* z,
                                   int n1, int n2)
{
    LAL_REQUIRE(c != nullptr && h != nullptr && r != nullptr && z != nullptr);
    LAL_REQUIRE(n1 >= 0 && n2 >= 0 && c == h->c);
    return precond<double>(h, r, z, n1, n2);
}

extern "C" int lal_pcg_solve_f64(lal_handle c, lal_hierarchy h, const double* b, double* x,
                                 const lal_solve_options* opts, lal_solve_info* info)
{
    LAL_REQUIRE(c != nullptr && h != nullptr && b != nullptr && x != nullptr && c == h->c);
    lal_solve_options o;
    lal_solve_default_options(&o);
    if(opts)
        o = *opts;
    LAL_REQUIRE(o.max_iter >= 0 && o.n1 >= 0 && o.n2 >= 0);
    LAL_REQUIRE(o.smoother >= 0 && o.smoother <= 6);
    return pcg<double>(h, b, x, h->res, h->z, h->p, h->q, o.rel_tol, o.abs_tol, o.max_iter,
                       o.n1, o.n2, info, nullptr, o.smoother);
}

extern "C" int lal_pcg_solve_op_f64(lal_handle c, lal_csrmv_descr descr, int m, int nnz,
                                    const int* rp, const int* ci, const double* v,
                                    lal_hierarchy h, const double* b, double* x,
                                    const lal_solve_options* opts, lal_solve_info* info)
{
    LAL_REQUIRE(c != nullptr && h != nullptr && b != nullptr && x != nullptr && c == h->c);
    LAL_REQUIRE(m == h->L[0].A.m && nnz >= 0 && rp != nullptr);
    LAL_REQUIRE(nnz == 0 || (ci != nullptr && v != nullptr));
    LAL_REQUIRE(descr == nullptr || (descr->m == m && descr->nnz == nnz));
    lal_solve_options o;
    lal_solve_default_options(&o);
    if(opts)
        o = *opts;
    LAL_REQUIRE(o.max_iter >= 0 && o.n1 >= 0 && o.n2 >= 0);
    LAL_REQUIRE(o.smoother >= 0 && o.smoother <= 6);
    // a non-owning view of the caller's matrix (never freed here)
    csr_dev A;
    A.m   = m;
    A.n   = m;
    A.nnz = nnz;
    A.rp  = const_cast<int*>(rp);
    A.ci  = const_cast<int*>(ci);
    A.v   = const_cast<double*>(v);
    A.d   = descr;
    return pcg<double>(h, b, x, h->res, h->z, h->p, h->q, o.rel_tol, o.abs_tol, o.max_iter,
                       o.n1, o.n2, info, &A, o.smoother);
}

extern "C" int lal_pcg_solve_mixed(lal_handle c, lal_hierarchy h, const double* b, double* x,
                                   const lal_solve_options* opts, lal_solve_info* info)
{
    LAL_REQUIRE(c != nullptr && h != nullptr && b != nullptr && x != nullptr && c == h->c);
    if(!h->has32)
    {
        lal::set_last_error("hierarchy was built without build_f32");
        return LAL_ERR_INVALID;
    }
    lal_solve_options o;
    lal_solve_default_options(&o);
    if(opts)
        o = *opts;
    LAL_REQUIRE(o.smoother == 0); // the FP32 levels run the Jacobi V-cycle only
    LAL_REQUIRE(o.max_iter >= 0 && o.n1 >= 0 && o.n2 >= 0);
    return pcg_mixed(h, b, x, o.rel_tol, o.abs_tol, o.max_iter, o.n1, o.n2, info);
}

extern "C" int lal_pcg_solve_reliable(lal_handle c, lal_hierarchy h, const double* b,
                                      double* x, const lal_solve_options* opts,
                                      lal_solve_info* info)
{
    LAL_REQUIRE(c != nullptr && h != nullptr && b != nullptr && x != nullptr && c == h->c);
    if(!h->has32)
    {
        lal::set_last_error("hierarchy was built without build_f32");
        return LAL_ERR_INVALID;
    }
    lal_solve_options o;
    lal_solve_default_options(&o);
    if(opts)
        o = *opts;
    LAL_REQUIRE(o.smoother == 0); // the FP32 levels run the Jacobi V-cycle only
    LAL_REQUIRE(o.max_iter >= 0 && o.n1 >= 0 && o.n2 >= 0);
    // without options the update threshold is 1e-2, which also holds the
    // iteration count on badly conditioned operators
    const double delta = opts ? o.inner_rel_tol : 1e-2;
    LAL_REQUIRE(delta > 0.0 && delta < 1.0);
    return pcg_reliable(h, b, x, o.rel_tol, o.abs_tol, o.max_iter, o.n1, o.n2, delta, info);
}

extern "C" int lal_ir_solve(lal_handle c, lal_hierarchy h, const double* b, double* x,
                            const lal_solve_options* opts, lal_solve_info* info)
{
    LAL_REQUIRE(c != nullptr && h != nullptr && b != nullptr && x != nullptr && c == h->c);
    if(!h->has32)
    {
        lal::set_last_error("hierarchy was built without build_f32");
        return LAL_ERR_INVALID;
    }
    lal_solve_options o;
    lal_solve_default_options(&o);
    if(opts)
        o = *opts;
    LAL_REQUIRE(o.smoother == 0); // the FP32 levels run the Jacobi V-cycle only
    const csr_dev& A = h->L[0].A;
    const int      n = A.m;
    double*        r = h->q; // FP64 outer residual lives in the FP64 q buffer
    LAL_TRY(lal::residual_f64(c, A.d, n, A.n, A.nnz, A.rp, A.ci, A.v, x, b, r));
    unsigned seq    = 0;
    double   init   = 0.0;
    LAL_TRY(lal::norm_partials<double>(c, n, r, h->part_r));
    LAL_TRY(post_norm(h, lal::PCG_BLOCKS, lal::S_RNORM0, &seq));
    LAL_TRY(wait_scalar(h, seq, lal::S_RNORM0, &init));
    double rn    = init;
    int    outer = 0, inner_total = 0;
    bool   conv  = false;
    while(true)
    {
        if(converges(rn, init, o.rel_tol, o.abs_tol))
        {
            conv = true;
            break;
        }
        if(outer >= o.max_outer)
            break;
        // inner FP32 solve of A d = r/|r|; level 0's FP32 rhs buffer is not
        // used by the V-cycle, so it holds the inner right-hand side
        float* rhs32 = h->L[0].w32.b;
        LAL_TRY(lal::scale_cast_f64_f32(c, n, r, 1.0 / rn, rhs32));
        LAL_HIP(hipMemsetAsync(h->d32, 0, sizeof(float) * n, c->stream));
        lal_solve_info ii{};
        LAL_TRY(pcg<float>(h, rhs32, h->d32, h->res32, h->z32, h->p32, h->q32,
                           o.inner_rel_tol, 1e-30, o.inner_max_iter, o.n1, o.n2, &ii));
        inner_total += ii.iterations + 1;
        // x += |r| d in FP64, then the true FP64 residual
        LAL_TRY(lal::axpy_f32_f64(c, n, rn, h->d32, x));
        LAL_TRY(lal::residual_f64(c, A.d, n, A.n, A.nnz, A.rp, A.ci, A.v, x, b, r));
        LAL_TRY(lal::norm_partials<double>(c, n, r, h->part_r));
        LAL_TRY(post_norm(h, lal::PCG_BLOCKS, lal::S_RNORM, &seq));
        LAL_TRY(wait_scalar(h, seq, lal::S_RNORM, &rn));
        outer++;
        if(std::isnan(rn))
            break;
    }
    if(info)
    {
        info->iterations       = inner_total;
        info->outer_iterations = outer;
        info->converged        = conv;
        info->initial_res_norm = init;
        info->final_res_norm   = rn;
    }
    return LAL_OK;
}

extern "C" int lal_adjoint_solve(lal_handle c, lal_hierarchy h, const double* g, double* lambda,
                                 int mixed, const lal_solve_options* opts, lal_solve_info* info)
{
    LAL_REQUIRE(c != nullptr && h != nullptr && g != nullptr && lambda != nullptr && c == h->c);
    LAL_REQUIRE(mixed >= 0 && mixed <= 3);
    LAL_HIP(hipMemsetAsync(lambda, 0, sizeof(double) * h->L[0].A.m, c->stream));
    if(mixed == 1)
        return lal_ir_solve(c, h, g, lambda, opts, info);
    if(mixed == 2)
        return lal_pcg_solve_mixed(c, h, g, lambda, opts, info);
    if(mixed == 3)
        return lal_pcg_solve_reliable(c, h, g, lambda, opts, info);
    return lal_pcg_solve_f64(c, h, g, lambda, opts, info);
}
