"""Transposes with a few long rows among short ones, bit for bit against the
oracle: rows of 129 to 256 entries, which a whole wavefront ranks while 16 lanes
take the short ones beside them, alone and several in a wavefront, the lengths on
either side, and longer rows, which the workgroup sorts in runs of 4096."""
import numpy as np
import pytest
import torch

from linalglib_amd import lal
from oracle.oracle import CSR
from tests.gpu_util import DevCSR, empty, host, log
from tests.test_gpu_amg import _gpu_transpose, csr_equal
from tests.test_gpu_transpose_counts import _column_lengths

pytestmark = pytest.mark.gpu

LENGTHS = {
    "one_a_wavefront": [n for k in (129, 160, 192, 193, 255, 256) for n in (k, 1, 0, 7) + (2,) * 28],
    "four_a_wavefront": [129, 256, 200, 130] * 2 + [1] * 400,
    "with_shorter_and_longer": [128, 129, 256, 257] + [257, 256, 300, 16] + [5] * 90 + [131],
}


@pytest.mark.parametrize("name", sorted(LENGTHS))
def test_long_rows_among_short_ones(oracle, name):
    log(f"transpose skewed {name}")
    lens = LENGTHS[name]
    assert sum(lens) <= 32 * len(lens)
    A = _column_lengths(lens, 700)
    want = oracle.transpose(A)
    h = lal.Handle()
    assert csr_equal(_gpu_transpose(h, A), want)
    d = DevCSR(A, f32=True)
    trp, tci = empty(A.n + 1, torch.int32), empty(A.nnz, torch.int32)
    tv = empty(A.nnz, torch.float32)
    lal.call("lal_transpose_f32", h.h, A.m, A.n, A.nnz, lal.ptr(d.row_ptr), lal.ptr(d.col_ind),
             lal.ptr(d.val), lal.ptr(trp), lal.ptr(tci), lal.ptr(tv))
    assert np.array_equal(host(trp), want.row_ptr) and np.array_equal(host(tci), want.col_ind)
    assert np.array_equal(host(tv), want.val.astype(np.float32))


def _time(h, rng, lens, m):
    """Fastest of seven transposes of a matrix whose columns have these lengths (us)."""
    lens = np.array(lens)
    col = np.repeat(np.arange(len(lens)), lens)
    row = rng.integers(0, m, len(col))
    order = np.lexsort((col, row))
    rp = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=m))])
    A = CSR(rp.astype(np.int32), col[order].astype(np.int32), rng.uniform(-1, 1, len(col)), m,
            len(lens))
    d = DevCSR(A)
    trp, tci = empty(A.n + 1, torch.int32), empty(A.nnz, torch.int32)
    tv = empty(A.nnz, torch.float64)
    times = []
    for _ in range(8):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        torch.cuda.synchronize()
        e[0].record()
        lal.call("lal_transpose_f64", h.h, A.m, A.n, A.nnz, lal.ptr(d.row_ptr),
                 lal.ptr(d.col_ind), lal.ptr(d.val), lal.ptr(trp), lal.ptr(tci), lal.ptr(tv))
        e[1].record()
        torch.cuda.synchronize()
        times.append(1e3 * e[0].elapsed_time(e[1]))
    return min(times[1:])


def test_long_rows_cost_no_more_than_their_entries():
    """2000 rows of 200 entries among 98,000 of 8, against 100,000 rows of 12: as
    many entries.  One lane's insertion sort per long row took 17 times as long
    (3170 us), the wavefronts' ranks 1.1 times."""
    h, rng = lal.Handle(), np.random.default_rng(2)
    even = _time(h, rng, [12] * 100000, 200000)
    skewed = _time(h, rng, ([200] + [8] * 49) * 2000, 200000)
    log(f"transpose of 1.2M entries: even rows {even:.0f} us, skewed {skewed:.0f} us")
    assert skewed <= 4 * even


HUBS = {
    "ends_of_runs": [257, 4095, 4096, 4097, 8191, 8192, 8193, 12289, 20000] + [3] * 900,
    "wavefront_rows": [300, 40, 5000, 60, 257, 33, 20000, 64],  # more than 32 on average
    "one_workgroup": [2, 300, 4100, 1, 0, 9000, 257, 130, 5] + [1] * 500,
}


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("name", sorted(HUBS))
def test_hubs(oracle, name, f32):
    log(f"transpose of hubs {name} f32={f32}")
    A = _column_lengths(HUBS[name], 20011)
    # the rows' columns in any order, as a caller may hold them
    rng = np.random.default_rng(1)
    row = np.repeat(np.arange(A.m), np.diff(A.row_ptr))
    order = np.lexsort((rng.random(A.nnz), row))
    A = CSR(A.row_ptr, A.col_ind[order], A.val[order].astype(np.float32).astype(np.float64), A.m, A.n)
    want, h, d = oracle.transpose(A), lal.Handle(), DevCSR(A, f32=f32)
    trp, tci, tv = empty(A.n + 1, torch.int32), empty(A.nnz, torch.int32), empty(A.nnz, d.dtype)
    lal.call("lal_transpose_f32" if f32 else "lal_transpose_f64", h.h, A.m, A.n, A.nnz,
             lal.ptr(d.row_ptr), lal.ptr(d.col_ind), lal.ptr(d.val), lal.ptr(trp), lal.ptr(tci),
             lal.ptr(tv))
    assert csr_equal((host(trp), host(tci), host(tv).astype(np.float64), A.n, A.m), want)


def test_hub_rows_with_repeated_columns(oracle):
    """Three entries of every row in the same column: they keep their order."""
    m = 3000
    ci = np.tile(np.array([1, 0, 1, 1, 2], np.int32), m)
    A = CSR(np.arange(0, 5 * m + 1, 5, dtype=np.int32), ci,
            np.random.default_rng(7).uniform(-1, 1, 5 * m), m, 4)
    log("transpose with repeated columns")
    assert csr_equal(_gpu_transpose(lal.Handle(), A), oracle.transpose(A))


def test_a_hub_costs_no_serial_sort():
    """One column of 40,000 entries among 100,000 of 12: one lane's insertion sort
    took seconds."""
    h, rng = lal.Handle(), np.random.default_rng(2)
    even = _time(h, rng, [12] * 103334, 200000)
    hub = _time(h, rng, [40000] + [12] * 100000, 200000)
    log(f"transpose of 1.24M entries: even rows {even:.0f} us, with a hub {hub:.0f} us")
    assert hub <= 50 * even
