"""The dense operator of the V-cycle's small end against the oracle's V-cycle: a
first level of 1023 and 1024 rows (the largest, an odd row length), of 1025 (the
next level down), of a handful of rows, a coarsest level of several rows (dense
inverse), unsmoothed aggregation; and the FP32 levels through the mixed solver."""
import numpy as np
import pytest
import torch

from linalglib_amd import lal, problems as pb
from oracle.oracle import CSR
from tests.gpu_util import DevCSR, dev, empty, host, log

pytestmark = pytest.mark.gpu

# name: (grid, rows of level 1, setup options)
CASES = {
    "rows1023": ((2896, 1), 1023, {}),
    "rows1024": ((2899, 1), 1024, {}),
    "rows1025": ((2902, 1), 1025, {}),
    "rows2": ((5, 1), 2, {}),
    "plane": ((64, 64), 949, {}),
    "two_levels_dense": ((64, 64), 949, {"max_levels": 2, "coarse_solver": 1}),
    "one_level_dense": ((64, 64), 949, {"max_levels": 1, "coarse_solver": 1}),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_cycle_operator(oracle, name):
    grid, rows, opts = CASES[name]
    rp, ci, v, m = pb.poisson2d(*grid)
    log(f"cycle operator {name}")
    h = lal.Handle()
    A = CSR(rp, ci, v, m, m)
    d = DevCSR(A)
    H = lal.Hierarchy(h, m, len(ci), d.row_ptr, d.col_ind, d.val, build_f32=1, **opts)
    assert H.dims(1, "A")[0] == rows
    rng = np.random.default_rng(3)
    x = rng.uniform(-1, 1, m)
    b = pb.rhs_from_solution(rp, ci, v, x)
    E = None
    if "max_levels" not in opts:
        ho = oracle.saamg_setup(A)
    else:  # the exact cycle of the same levels, pinned to the oracle elsewhere
        E = lal.Hierarchy(h, m, len(ci), d.row_ptr, d.col_ind, d.val, exact=1, **opts)
    for r in (rng.uniform(-1, 1, m), b):
        z, ref = empty(m, torch.float64), empty(m, torch.float64)
        H.precond(dev(r), z)
        if E is None:
            ref = ho.precond(r, 1, 1, 1)
        else:
            E.precond(dev(r), ref)
            ref = host(ref)
        # the bar of the other fast V-cycles against the oracle
        assert np.linalg.norm(host(z) - ref) <= 1e-10 * np.linalg.norm(ref)
    for solve in ("pcg", "pcg_mixed"):
        X = torch.zeros(m, dtype=torch.float64, device="cuda")
        info = getattr(H, solve)(dev(b), X, rel_tol=1e-9, abs_tol=1e-300, max_iter=400)
        assert info.converged
        got = b - pb.rhs_from_solution(rp, ci, v, host(X))
        # the recursive norm meets 1e-9; the true one may differ by rounding
        assert np.abs(got).max() <= 2e-9 * np.abs(b).max()


def test_cycle_operator_unsmoothed(oracle):
    rp, ci, v, m = pb.poisson3d(12)
    A = CSR(rp, ci, v, m, m)
    h = lal.Handle()
    d = DevCSR(A)
    log("cycle operator, unsmoothed aggregation")
    H = lal.Hierarchy(h, m, len(ci), d.row_ptr, d.col_ind, d.val, unsmoothed=True)
    E = lal.Hierarchy(h, m, len(ci), d.row_ptr, d.col_ind, d.val, unsmoothed=True, exact=1)
    r = np.random.default_rng(4).uniform(-1, 1, m)
    z, ref = empty(m, torch.float64), empty(m, torch.float64)
    H.precond(dev(r), z)
    E.precond(dev(r), ref)
    ref = host(ref)
    assert np.linalg.norm(host(z) - ref) <= 1e-10 * np.linalg.norm(ref)
