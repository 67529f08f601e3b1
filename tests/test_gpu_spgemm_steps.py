"""The sparse product's lane layouts, bit for bit against the oracle: rows of A
and B at the edges of the lane groups (8, 16, 32 and 64 lanes), B rows of one
and of several steps, launches of few rows (which load a batch ahead) and of
many, products that are subnormal, -0.0 or cancel exactly."""
import numpy as np
import pytest

from linalglib_amd import lal
from oracle.oracle import CSR
from tests.gpu_util import log
from tests.test_gpu_amg import _gpu_spgemm, csr_equal

pytestmark = pytest.mark.gpu


def _matrix(rng, m, n, low, high):
    """Rows of `low` or `high` entries (mostly low), values of several scales."""
    lens = np.where(rng.random(m) < 0.1, high, low)
    lens[rng.integers(0, m, m // 50)] = 0
    rp = np.zeros(m + 1, np.int32)
    rp[1:] = np.cumsum(lens)
    # distinct ascending columns per row: a random start and random gaps
    ci = np.empty(rp[-1], np.int32)
    for i in range(m):
        ci[rp[i]:rp[i + 1]] = np.sort(rng.choice(n, size=lens[i], replace=False))
    v = rng.choice([1.0, -1.0, 0.0, -0.0, 3e-160, -2.5e-160, 0.1], size=rp[-1])
    v = np.where(rng.random(rp[-1]) < 0.5, v, rng.uniform(-1, 1, rp[-1]))
    return CSR(rp, ci, v, m, n)


# (rows of A, entries per A row, entries per B row): the mean lengths pick the
# lanes per row, the longer rows cross the chunk and step bounds
@pytest.mark.parametrize("m,alen,blen", [
    (50, (3, 9), (2, 9)),        # few rows: a wavefront each, 8 steps side by side
    (70, (40, 130), (9, 17)),    # several chunks of 64 A entries
    (60, (20, 65), (60, 200)),   # one step at a time, B rows of several steps
    (60, (20, 64), (30, 33)),    # 32 lanes per B row
    (40000, (3, 8), (3, 8)),     # many rows: 8 lanes each
    (20000, (12, 17), (6, 9)),   # 16 lanes, two steps side by side
    (9000, (25, 33), (12, 17)),  # 32 lanes, 16 per B row
    (5000, (50, 70), (20, 40)),  # a wavefront without loading ahead
])
def test_steps_and_lanes(oracle, m, alen, blen):
    rng = np.random.default_rng(m + alen[0])
    k = 400
    A = _matrix(rng, m, k, *alen)
    log(f"spgemm steps m={m} A rows {alen} B rows {blen}")
    h = lal.Handle()
    for n in (250, 3000):
        B = _matrix(rng, k, n, *blen)
        assert csr_equal(_gpu_spgemm(h, A, B), oracle.csrgemm(A, B))
