"""Products of matrices with many long rows among more short ones: the lanes per
row follow the mean length, the tables each row's own, and every launch keeps its
tables within a workgroup's share of LDS; bit for bit against the oracle."""
import numpy as np
import pytest

from linalglib_amd import lal, problems as pb
from oracle.oracle import CSR
from tests.gpu_util import log
from tests.test_gpu_amg import _gpu_spgemm, csr_equal

pytestmark = pytest.mark.gpu

K = 4001  # (a prime: the multiples of a step are distinct)


def _spread(rows, length, n, rng):
    """rows x length distinct columns below n (a prime), ascending."""
    start, step = rng.integers(0, n, (rows, 1)), rng.integers(1, n, (rows, 1))
    return np.sort((start + step * np.arange(length)) % n, axis=1)


def _skewed(m, long_rows, length, rng):
    """m rows, the last `long_rows` odd ones of `length` entries, the others empty."""
    lens = np.zeros(m, np.int64)
    lens[m - 2 * long_rows + 1::2] = length
    rp = np.zeros(m + 1, np.int32)
    rp[1:] = np.cumsum(lens)
    ci = _spread(long_rows, length, K, rng).ravel()
    return CSR(rp, ci.astype(np.int32), rng.uniform(-1, 1, len(ci)), m, K)


# mean lengths of A that give 8 and 16 lanes per row; rows enough that a launch
# of so many lanes each is not one of few rows
@pytest.mark.parametrize("m,long_rows,length,slots", [
    (180000, 33000, 36, 1024), (290000, 33000, 70, 2048), (580000, 33000, 140, 4096),
    (80000, 16500, 70, 2048), (160000, 16500, 140, 4096)])
def test_long_rows_among_short_ones(oracle, m, long_rows, length, slots):
    log(f"spgemm skewed: {long_rows} of {m} rows with {length} entries")
    rng = np.random.default_rng(length)
    A = _skewed(m, long_rows, length, rng)
    n = 60013
    B = CSR(np.arange(0, 8 * K + 1, 8, dtype=np.int32),
            _spread(K, 8, n, rng).ravel().astype(np.int32), rng.uniform(-1, 1, 8 * K), K, n)
    C = oracle.csrgemm(A, B)
    per_row = np.diff(C.row_ptr)
    most = np.median(per_row[per_row > 0])
    lanes = 8 if A.nnz <= 8 * m else 16
    assert slots // 4 < most <= slots // 2 and (per_row > slots // 4).sum() * lanes >= 262144
    assert csr_equal(_gpu_spgemm(lal.Handle(), A, B), C)


@pytest.mark.parametrize("k,tables", [(4, 128), (9, 512), (14, 1024)])
def test_counting_lanes(oracle, k, tables):
    """Square products of graphs on either side of the line where the counting pass
    doubles its lanes (8 lanes a row and 128 slots; 16 and 512 or 1024)."""
    n = 34000
    rp, ci, m, edges, entry, edge, sign, dpos = pb.knn_laplacian(n, k=k, seed=3)
    v = np.random.default_rng(k).uniform(-1, 1, len(ci))
    A = CSR(rp, ci, v, m, m)
    products = np.add.reduceat(np.diff(rp)[ci], rp[:-1])
    log(f"counting lanes: {len(ci) / m:.1f} per row, {products.mean():.0f} products")
    assert tables // 2 < 2 * np.median(products) <= tables
    assert csr_equal(_gpu_spgemm(lal.Handle(), A, A), oracle.csrgemm(A, A))
