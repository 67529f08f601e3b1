"""PCG's direction formed inside the product (finest levels of up to 262,144 rows)
against the separate pass: the same solve through a caller's operator, aligned
(also formed inside) and at an odd element offset (separate kernels), and sizes
around the limit; FP64, FP32 refinement and reliable updates, one and many blocks."""
import numpy as np
import pytest
import torch

from linalglib_amd import lal, problems as pb
from oracle.oracle import CSR
from tests.gpu_util import DevCSR, dev, host, log

pytestmark = pytest.mark.gpu


def _odd(t):
    """A copy of t that starts one element off its allocation."""
    big = torch.zeros(t.numel() + 1, dtype=t.dtype, device="cuda")
    big[1:] = t
    return big[1:]


@pytest.mark.parametrize("grid", [(5, 3), (64, 63), (256, 255), (512, 512), (512, 513)])
def test_direction_in_the_product(grid):
    rp, ci, v, m = pb.poisson2d(*grid)
    log(f"direction in the product, {m} rows")
    h = lal.Handle()
    d = DevCSR(CSR(rp, ci, v, m, m))
    H = lal.Hierarchy(h, m, len(ci), d.row_ptr, d.col_ind, d.val, build_f32=1)
    b = pb.rhs_from_solution(rp, ci, v, np.random.default_rng(8).uniform(-1, 1, m))
    kw = dict(rel_tol=1e-9, abs_tol=1e-300, max_iter=300)

    def solve(f, *a):
        X = torch.zeros(m, dtype=torch.float64, device="cuda")
        info = f(*a, dev(b), X, **kw)
        assert info.converged
        res = b - pb.rhs_from_solution(rp, ci, v, host(X))
        # the recursive norm meets 1e-9; the true one may differ by rounding
        assert np.abs(res).max() <= 2e-9 * np.abs(b).max()
        return host(X), info.iterations

    x, it = solve(H.pcg)
    same = lal.CsrDescr(h, m, m, len(ci), d.row_ptr, d.col_ind)
    xa, ita = solve(H.pcg_op, (d.row_ptr, d.col_ind, d.val, m, len(ci), same))
    assert ita == it and np.array_equal(xa, x)
    off = (d.row_ptr, _odd(d.col_ind), _odd(d.val), m, len(ci))
    odd = lal.CsrDescr(h, m, m, len(ci), off[0], off[1])
    # (other block sums in the inner products)
    _, ito = solve(H.pcg_op, off + (odd,))
    assert abs(ito - it) <= 1
    for f in (H.pcg_reliable, H.pcg_mixed, H.ir):
        solve(f)
