"""Setup passes with 8, 16 and 64 lanes per row on rows at and beyond what the
lanes keep in registers (4 entries each), the transpose's sorts likewise, and
the one-launch scan at its tile and size edges; bit for bit against the oracle."""
import ctypes as C

import numpy as np
import pytest
import torch

from linalglib_amd import lal
from oracle.oracle import CSR
from tests.gpu_util import DevCSR, dev, empty, host, log
from tests.test_gpu_amg import _gpu_transpose, csr_equal

pytestmark = pytest.mark.gpu


def _matrix(m, usual, rare, seed):
    """Square, diagonal in every row, mostly `usual` entries per row and now
    and then one of `rare`."""
    rng = np.random.default_rng(seed)
    lens = np.full(m, usual)
    lens[rng.choice(m, len(rare) * 3, replace=False)] = np.repeat(rare, 3)
    rows = []
    for i in range(m):
        c = rng.choice(m, size=lens[i], replace=False)
        rows.append(np.unique(np.append(c[c != i][: lens[i] - 1], i)))
    rp = np.zeros(m + 1, np.int32)
    rp[1:] = np.cumsum([len(r) for r in rows])
    ci = np.concatenate(rows).astype(np.int32)
    v = rng.uniform(-1, 0, rp[-1])
    v[ci == np.repeat(np.arange(m), np.diff(rp))] = 3.0
    return CSR(rp, ci, v, m, m)


@pytest.mark.parametrize("usual,rare", [
    (5, (8, 9, 31, 32, 33, 70)),          # 8 lanes keep 32 entries
    (20, (16, 63, 64, 65, 130)),          # 16 lanes keep 64
    (60, (64, 255, 256, 257, 400)),       # a wavefront keeps 256
])
def test_strength_pmis_prolongator_transpose(oracle, usual, rare):
    A = _matrix(700, usual, rare, usual)
    m, nnz, d, h = A.m, A.nnz, DevCSR(A), lal.Handle()
    for eps in (0.05, 0.2):
        log(f"setup lanes: rows of {usual}, some of {rare}, eps {eps}")
        conn = empty(nnz, torch.int32)
        lal.call("lal_sa_strength_f64", h.h, m, nnz, lal.ptr(d.row_ptr), lal.ptr(d.col_ind),
                 lal.ptr(d.val), eps, lal.ptr(conn))
        c_ref = oracle.strength(A, eps)
        assert np.array_equal(host(conn), c_ref)
        agg = empty(m, torch.int64)
        lal.call("lal_pmis_aggregate", h.h, m, nnz, lal.ptr(d.row_ptr), lal.ptr(d.col_ind),
                 lal.ptr(conn), lal.ptr(agg))
        a_ref = oracle.aggregates(A, c_ref)
        assert np.array_equal(host(agg), a_ref)
        # the true aggregates, and many (a long list of columns per row)
        for ids in (a_ref, np.where(np.arange(m) % 7 == 3, -2, np.arange(m) // 2)):
            ids = ids.astype(np.int64)
            prp, D = empty(m + 1, torch.int32), dev(ids, np.int64)
            n_p, nc = C.c_int(), C.c_int()
            lal.call("lal_sa_prolongator_nnz", h.h, m, nnz, lal.ptr(d.row_ptr),
                     lal.ptr(d.col_ind), lal.ptr(conn), lal.ptr(D), lal.ptr(prp), C.byref(n_p),
                     C.byref(nc))
            ref = oracle.prolongator(A, c_ref, ids)
            assert (n_p.value, nc.value) == (ref.nnz, ref.n)
            pci, pv = empty(n_p.value, torch.int32), empty(n_p.value, torch.float64)
            lal.call("lal_sa_prolongator_fill_f64", h.h, m, nnz, lal.ptr(d.row_ptr),
                     lal.ptr(d.col_ind), lal.ptr(d.val), lal.ptr(conn), lal.ptr(D), 2.0 / 3.0,
                     lal.ptr(prp), lal.ptr(pci), lal.ptr(pv))
            got = (host(prp), host(pci)[: ref.nnz], host(pv)[: ref.nnz], m, nc.value)
            assert csr_equal(got, ref)
    assert csr_equal(_gpu_transpose(h, A), oracle.transpose(A))
    # its transpose has rows of other lengths
    T = oracle.transpose(A)
    assert csr_equal(_gpu_transpose(h, T), oracle.transpose(T))


@pytest.mark.parametrize("n", [1, 7, 2047, 2048, 2049, 4096, 16383, 16384, 16385, 70000])
def test_scan_sizes(n):
    h = lal.Handle()
    x = np.random.default_rng(n).integers(-5, 9, n)
    for name, dt in (("lal_exclusive_scan_i32", np.int32), ("lal_exclusive_scan_i64", np.int64)):
        X = dev(x, dt)
        lal.call(name, h.h, n, lal.ptr(X))
        assert np.array_equal(host(X), np.concatenate([[0], np.cumsum(x)[:-1]]))
