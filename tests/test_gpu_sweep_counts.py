"""The fast V-cycle with no, two or three pre-sweeps against the oracle's, on
operators whose coarse levels gather x by column lists (blocks that span less
and more than 65536 columns) and on ones that do not; and the solvers with two
sweeps on either side, whose FP32 levels take the same path."""
import numpy as np
import pytest
import torch

from linalglib_amd import lal, problems as pb
from oracle.oracle import CSR
from tests.gpu_util import DevCSR, dev, empty, host, log
from tests.test_gpu_vcycle_operators import CASES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", sorted(CASES))
def test_sweep_counts(oracle, name):
    rp, ci, v, m = CASES[name]()
    d = DevCSR(CSR(rp, ci, v, m, m))
    H = lal.Hierarchy(lal.Handle(), m, len(ci), d.row_ptr, d.col_ind, d.val)
    ho = oracle.saamg_setup(CSR(rp, ci, v, m, m))
    r = np.random.default_rng(5).uniform(-1, 1, m)
    R, z = dev(r), empty(m, torch.float64)
    for n1 in (0, 2, 3):
        for n2 in (0, 1, 2):
            log(f"sweep counts {name} n1={n1} n2={n2}")
            H.precond(R, z, n1, n2)
            ref = ho.precond(r, n1, n2, 1)
            # the bar of the other fast V-cycles against the oracle
            assert np.linalg.norm(host(z) - ref) <= 1e-10 * np.linalg.norm(ref)


@pytest.mark.parametrize("solve", ["pcg", "pcg_mixed", "pcg_reliable", "ir"])
@pytest.mark.parametrize("name", ["grid33", "lines_far", "long_row"])
def test_solvers_with_two_sweeps(name, solve):
    rp, ci, v, m = CASES[name]()
    log(f"two sweeps {name} {solve}")
    d = DevCSR(CSR(rp, ci, v, m, m))
    H = lal.Hierarchy(lal.Handle(), m, len(ci), d.row_ptr, d.col_ind, d.val, build_f32=1)
    b = pb.rhs_from_solution(rp, ci, v, np.random.default_rng(6).uniform(-1, 1, m))
    X = torch.zeros(m, dtype=torch.float64, device="cuda")
    info = getattr(H, solve)(dev(b), X, rel_tol=1e-9, abs_tol=1e-300, max_iter=400, n1=2, n2=2)
    assert info.converged
    got = b - pb.rhs_from_solution(rp, ci, v, host(X))
    # the recursive norm meets 1e-9; the true one may differ by rounding
    assert np.abs(got).max() <= 2e-9 * np.abs(b).max()
