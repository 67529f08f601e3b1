"""Hierarchies whose levels are built by one workgroup, bit for bit against the
oracle's: at and beyond the limits of each lane count (1024 rows of up to 11
entries, 512 of 12 to 47, 128 of 48 and more; 8192 entries), rows in any column
order, without a diagonal, alone, or empty; smoothed and unsmoothed.  And sparse
products planned by one workgroup, at its chunk and row limits, with rows whose
tables lie in global memory."""
import numpy as np
import pytest
import scipy.sparse as sp

from linalglib_amd import lal, problems as pb
from oracle.oracle import CSR
from tests.gpu_util import DevCSR, log
from tests.test_gpu_amg import _gpu_spgemm, csr_equal

pytestmark = pytest.mark.gpu


def _csr(S):
    return CSR(S.indptr.astype(np.int32), S.indices.astype(np.int32), S.data.astype(float),
               *S.shape)


def _band(m, half):
    """Symmetric band of about 2 * half + 1 entries per row, M-matrix."""
    rng = np.random.default_rng(m * 7 + half)
    i, j = np.where(np.abs(np.subtract.outer(np.arange(m), np.arange(m))) <= half)
    up = i < j
    # one coupling in ten is strong
    w = np.where(rng.random(up.sum()) < 0.1, rng.uniform(2, 5, up.sum()),
                 rng.uniform(0.001, 0.01, up.sum()))
    S = sp.coo_matrix((-w, (i[up], j[up])), (m, m)).tocsr()
    S = S + S.T
    return (S + sp.diags(-np.asarray(S.sum(axis=1)).ravel() + 0.01)).tocsr()


def _odd_rows():
    """Columns in random order; a row alone, an empty one, one without diagonal."""
    S = _band(200, 3).tolil()
    S[17, :], S[:, 17] = 0.0, 0.0
    S[17, 17] = 2.0
    S[40, :], S[:, 40] = 0.0, 0.0
    S[90, 90] = 0.0
    S = S.tocsr()
    S.eliminate_zeros()
    rng = np.random.default_rng(1)
    for r in range(S.shape[0]):
        a, b = S.indptr[r], S.indptr[r + 1]
        o = rng.permutation(b - a) + a
        S.indices[a:b], S.data[a:b] = S.indices[o], S.data[o]
    return _csr(S)


def _chain(m):
    rp, ci, v, n = pb.poisson2d(m, 1)
    return CSR(rp, ci, v, n, n)


CASES = {
    "rows1": lambda: CSR(np.array([0, 1], np.int32), np.array([0], np.int32), np.array([2.0]), 1, 1),
    "rows2": lambda: _chain(2),
    "rows1024": lambda: _chain(1024),
    "rows1025": lambda: _chain(1025),
    "lanes16_512": lambda: _csr(_band(512, 7)),
    "lanes16_513": lambda: _csr(_band(513, 7)),
    "lanes64_128": lambda: _csr(_band(128, 31)),
    "lanes64_129": lambda: _csr(_band(129, 31)),
    "full90": lambda: _csr(_band(90, 90)),   # 8100 entries
    "full91": lambda: _csr(_band(91, 91)),   # 8281
    "odd_rows": _odd_rows,
}


def _equal(got, ref):
    """Bit for bit; a NaN (odd_rows: 1/0 in P) only by its place, since the sign
    that inf - inf gives it is the processor's."""
    rp, ci, v, m, n = got
    both = np.isnan(v) & np.isnan(ref.val) if v.shape == ref.val.shape else np.zeros(0, bool)
    clean = CSR(ref.row_ptr, ref.col_ind, np.where(both, 0.0, ref.val), ref.m, ref.n) \
        if len(both) else ref
    return csr_equal((rp, ci, np.where(both, 0.0, v) if len(both) else v, m, n), clean)


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("unsmoothed", [False, True])
def test_small_levels(oracle, name, unsmoothed):
    A = CASES[name]()
    log(f"small levels {name} unsmoothed={unsmoothed}")
    ho = oracle.uaamg_setup(A) if unsmoothed else oracle.saamg_setup(A)
    h, d = lal.Handle(), DevCSR(A)
    # (exact: an operator without a diagonal entry has no fast inverse)
    H = lal.Hierarchy(h, A.m, A.nnz, d.row_ptr, d.col_ind, d.val, unsmoothed=unsmoothed, exact=1,
                      coarse_solver=0)
    assert H.levels == ho.levels
    for l in range(H.levels + 1):
        for kind in ("A",) if l == H.levels else ("A", "P", "R"):
            assert _equal(H.level(l, kind), ho.get(l, kind)), (l, kind)


def _sparse(m, n, per_row, heavy, seed):
    rng = np.random.default_rng(seed)
    lens = np.full(m, per_row)
    lens[rng.integers(0, m, max(1, m // 100))] = 0
    for r, k in heavy:
        lens[r] = k
    rp = np.zeros(m + 1, np.int32)
    rp[1:] = np.cumsum(lens)
    ci = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lens])
    return CSR(rp, ci.astype(np.int32), rng.uniform(-1, 1, rp[-1]), m, n)


@pytest.mark.parametrize("m", [1, 1023, 1024, 1025, 16383, 16384])
def test_planned_products(oracle, m):
    log(f"planned products m={m}")
    k, n = 3000, 20000
    # the last row's product has far more entries than a table in LDS holds
    A = _sparse(m, k, 3, [(m - 1, 2500)], m)
    B = _sparse(k, n, 6, [(7, 900)], 5)
    h = lal.Handle()
    assert csr_equal(_gpu_spgemm(h, A, B), oracle.csrgemm(A, B))
