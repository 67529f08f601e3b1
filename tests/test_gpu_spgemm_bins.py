"""Products whose rows fall into every table size, few enough that the sizes share
a launch and more than one launch takes, bit for bit against the oracle."""
import numpy as np
import pytest

from linalglib_amd import lal
from oracle.oracle import CSR
from tests.gpu_util import log
from tests.test_gpu_amg import _gpu_spgemm, csr_equal

pytestmark = pytest.mark.gpu


def _csr(lens, n, seed):
    rng = np.random.default_rng(seed)
    rp = np.zeros(len(lens) + 1, np.int32)
    rp[1:] = np.cumsum(lens)
    ci = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lens])
    return CSR(rp, ci.astype(np.int32), rng.uniform(-1, 1, rp[-1]), len(lens), n)


@pytest.mark.parametrize("m", [8, 300, 7000])
def test_rows_of_every_table_size(oracle, m):
    log(f"spgemm bins m={m}")
    # rows of C of about 3 * length columns: tables of 64 to 4096 slots
    lens = np.resize([1, 9, 20, 42, 85, 170, 340, 600], m)
    A, B = _csr(lens, 2500, m), _csr(np.full(2500, 3), 40000, 1)
    C = oracle.csrgemm(A, B)
    per_row = np.diff(C.row_ptr)
    assert per_row.min() <= 3 and 1024 < per_row.max() <= 2048
    assert csr_equal(_gpu_spgemm(lal.Handle(), A, B), C)
