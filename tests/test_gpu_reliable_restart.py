"""The reliable-update solve near FP32's limit: on face diffusion 96^3 to 1e-12 its
recurrence can drift above the last true residual, where it stayed for thousands of
steps (seed 18: more than 9000 for most right-hand sides) until an interval far
longer than those before became an update with a restart.  A dozen right-hand sides
that differ by rounding: the drift itself depends on every bit."""
import numpy as np
import pytest
import torch

from linalglib_amd import lal, problems as pb
from tests.gpu_util import dev, host, log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [17, 18])
def test_drifting_recurrence_restarts(seed):
    rp, ci, m, nf, entry, face, sign = pb.diffusion_faces(96)
    rng = np.random.default_rng(seed)
    v = pb.assemble_faces(len(ci), entry, face, sign, np.exp(rng.standard_normal(nf)))
    b, xt = rng.standard_normal(m), rng.standard_normal(m)
    H = lal.Hierarchy(lal.Handle(), m, len(ci), dev(rp), dev(ci), dev(v), build_f32=1)
    X = torch.zeros(m, dtype=torch.float64, device="cuda")
    assert H.pcg(dev(b), X, rel_tol=1e-13, abs_tol=1e-300, max_iter=300).converged
    x, its = host(X), []
    for k in range(12):
        g = x - xt * (1 + 1e-13 * rng.standard_normal(m))
        Y = torch.zeros(m, dtype=torch.float64, device="cuda")
        # about 370 steps without a drift, of at most four times the longest
        # interval (60); an order of magnitude below the unbounded drifts
        info = H.pcg_reliable(dev(g), Y, rel_tol=1e-12, abs_tol=1e-300, max_iter=1500)
        its.append(info.iterations)
        assert info.converged, its
        if k == 0:
            res = g - pb.rhs_from_solution(rp, ci, v, host(Y))
            # (the solver's own residual is the true one, in another order of sums)
            assert np.abs(res).max() <= 1.1e-12 * np.abs(g).max()
    log(f"reliable restart, seed {seed}: steps {sorted(its)}")
