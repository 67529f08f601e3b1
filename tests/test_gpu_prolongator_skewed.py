"""The prolongator of matrices with a few long rows among short ones, which take a
wavefront each whatever the mean length gives the others: bit for bit against the
oracle with several such rows beside each other, and in no more time than where
every row takes a wavefront."""
import ctypes as C
import time

import numpy as np
import pytest
import torch

from linalglib_amd import lal
from oracle.oracle import CSR
from tests.gpu_util import DevCSR, dev, empty, host, log
from tests.test_gpu_amg import csr_equal

pytestmark = pytest.mark.gpu


def _matrix(lens, seed):
    """Square, row i with lens[i] entries, the diagonal among them."""
    m, rng = len(lens), np.random.default_rng(seed)
    rows = [np.sort(np.append(rng.choice(m - 1, k - 1, replace=False), m - 1)) for k in lens]
    rows = [(r + 1 + i) % m for i, r in enumerate(rows)]  # (m - 1 becomes i)
    rp = np.zeros(m + 1, np.int32)
    rp[1:] = np.cumsum(lens)
    ci = np.concatenate([np.sort(r) for r in rows]).astype(np.int32)
    v = rng.uniform(-1, 0, rp[-1])
    v[ci == np.repeat(np.arange(m), lens)] = 3.0
    return CSR(rp, ci, v, m, m)


def _prolongator(h, A, d, conn, agg):
    prp, n_p, nc = empty(A.m + 1, torch.int32), C.c_int(), C.c_int()
    lal.call("lal_sa_prolongator_nnz", h.h, A.m, A.nnz, lal.ptr(d.row_ptr), lal.ptr(d.col_ind),
             lal.ptr(conn), lal.ptr(agg), lal.ptr(prp), C.byref(n_p), C.byref(nc))
    pci, pv = empty(n_p.value, torch.int32), empty(n_p.value, torch.float64)
    lal.call("lal_sa_prolongator_fill_f64", h.h, A.m, A.nnz, lal.ptr(d.row_ptr),
             lal.ptr(d.col_ind), lal.ptr(d.val), lal.ptr(conn), lal.ptr(agg), 2.0 / 3.0,
             lal.ptr(prp), lal.ptr(pci), lal.ptr(pv))
    return prp, pci, pv, n_p.value, nc.value


@pytest.mark.parametrize("lens", [
    [3] * 400 + [33, 34, 200, 300, 32, 33] + [4] * 300 + [90],           # 8 lanes keep 32
    [15] * 400 + [65, 66, 300, 500, 64, 65, 256, 257] + [13] * 300 + [400],  # 16 keep 64
], ids=["8_lanes", "16_lanes"])
def test_long_rows_among_short_ones(oracle, lens):
    A = _matrix(lens, len(lens))
    log(f"prolongator skewed: {A.m} rows, {A.nnz} entries")
    h, d = lal.Handle(), DevCSR(A)
    conn_ref = oracle.strength(A, 0.05)
    for ids in (oracle.aggregates(A, conn_ref), np.arange(A.m) // 2):
        ids = ids.astype(np.int64)
        prp, pci, pv, n, nc = _prolongator(h, A, d, dev(conn_ref, np.int32), dev(ids, np.int64))
        ref = oracle.prolongator(A, conn_ref, ids)
        assert (n, nc) == (ref.nnz, ref.n)
        assert csr_equal((host(prp), host(pci)[:n], host(pv)[:n], A.m, nc), ref)


def test_long_rows_take_a_wavefront_each():
    """50 rows of 1000 entries among 3950 of 20 (16 lanes a row), against the same
    among rows of 50 (a wavefront a row): with 16 lanes for the long rows too the
    former took more than three times as long, for fewer entries."""
    h, took = lal.Handle(), []
    for usual in (20, 50):
        lens = np.full(4000, usual)
        lens[40::80] = 1000
        A = _matrix(lens, 3)
        d = DevCSR(A)
        conn, agg = empty(A.nnz, torch.int32) + 1, dev(np.arange(A.m) // 2, np.int64)
        best = np.inf
        for _ in range(6):
            torch.cuda.synchronize()
            t = time.perf_counter()
            _prolongator(h, A, d, conn, agg)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t)
        took.append(1e6 * best)
    log(f"prolongator: {took[0]:.0f} us among rows of 20, {took[1]:.0f} us among rows of 50")
    assert took[0] <= 1.5 * took[1]
