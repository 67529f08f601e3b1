"""The transpose's column counts through a workgroup's table and its row sorts,
bit for bit against the oracle: every column distinct (a permutation, a full
table), one column for all entries, columns that share table slots, entry counts
around the workgroup's 2048, and rows around the 128 entries that 16 lanes keep."""
import numpy as np
import pytest

from linalglib_amd import lal
from oracle.oracle import CSR
from tests.gpu_util import log
from tests.test_gpu_amg import _gpu_transpose, csr_equal

pytestmark = pytest.mark.gpu


def _rows(cols, n, seed):
    """CSR whose row i holds the columns cols[i]."""
    rp = np.zeros(len(cols) + 1, np.int32)
    rp[1:] = np.cumsum([len(c) for c in cols])
    ci = np.concatenate(cols).astype(np.int32)
    return CSR(rp, ci, np.random.default_rng(seed).uniform(-1, 1, len(ci)), len(cols), n)


def _permutation(m):
    return _rows([[c] for c in np.random.default_rng(m).permutation(m)], m, 1)


def _spaced(m, step):
    return _rows([[(i * step) % (m * step)] for i in range(m)], m * step, 2)


def _column_lengths(lens, m):
    """Column c has lens[c] entries, spread over the rows."""
    rng = np.random.default_rng(3)
    rows = [[] for _ in range(m)]
    for c, k in enumerate(lens):
        for i in rng.choice(m, k, replace=False):
            rows[i].append(c)
    return _rows([np.array(sorted(r), int) for r in rows], len(lens), 4)


CASES = {
    "permutation_2047": lambda: _permutation(2047),
    "permutation_2048": lambda: _permutation(2048),
    "permutation_5001": lambda: _permutation(5001),
    "one_column": lambda: _rows([[0]] * 5000, 3, 5),
    "spaced_4096": lambda: _spaced(3000, 4096),
    "lengths_short": lambda: _column_lengths([1, 2, 15, 16, 17, 127, 128, 129, 200] + [9] * 400, 900),
    "lengths_long": lambda: _column_lengths([40, 63, 64, 65, 255, 256, 257] * 6, 900),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_transpose_counts(oracle, name):
    A = CASES[name]()
    log(f"transpose counts {name}")
    assert csr_equal(_gpu_transpose(lal.Handle(), A), oracle.transpose(A))
