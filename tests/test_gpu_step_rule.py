"""PCG on either side of the lines where it forms its direction inside the product
(two million entries; 706,000 where rows hold more than 13): the same solve through
a caller's operator, bit for bit, and through one at an odd element offset, which
takes the separate kernels."""
import numpy as np
import pytest
import torch

from linalglib_amd import lal, problems as pb
from oracle.oracle import CSR
from tests.gpu_util import DevCSR, dev, host, log
from tests.test_gpu_step_product import _odd

pytestmark = pytest.mark.gpu


def _graph(n):
    rp, ci, m, edges, entry, edge, sign, dpos = pb.knn_laplacian(n, seed=4)
    w = np.exp(0.5 * np.random.default_rng(4).standard_normal(len(edges)))
    v = np.bincount(entry, weights=sign * w[edge], minlength=len(ci))
    v[dpos] += 1e-2
    return rp, ci, v, m


CASES = {"grid_below": lambda: pb.poisson2d(700, 599), "grid_above": lambda: pb.poisson2d(700, 601),
         "graph_below": lambda: _graph(47500), "graph_above": lambda: _graph(48500)}


@pytest.mark.parametrize("name", sorted(CASES))
def test_either_side(name):
    rp, ci, v, m = CASES[name]()
    nnz = len(ci)
    line = 2 << 20 if nnz <= 13 * m else 706000
    assert (nnz <= line) == name.endswith("below")
    log(f"step rule {name}: {m} rows, {nnz} entries")
    h = lal.Handle()
    d = DevCSR(CSR(rp, ci, v, m, m))
    H = lal.Hierarchy(h, m, nnz, d.row_ptr, d.col_ind, d.val)
    b = pb.rhs_from_solution(rp, ci, v, np.random.default_rng(8).uniform(-1, 1, m))
    off = _odd(d.col_ind), _odd(d.val)
    ops = [None, (d.col_ind, d.val), off]
    xs, its = [], []
    for o in ops:
        X = torch.zeros(m, dtype=torch.float64, device="cuda")
        kw = dict(rel_tol=1e-9, abs_tol=1e-300, max_iter=300)
        if o is None:
            info = H.pcg(dev(b), X, **kw)
        else:
            descr = lal.CsrDescr(h, m, m, nnz, d.row_ptr, o[0])
            info = H.pcg_op((d.row_ptr, *o, m, nnz, descr), dev(b), X, **kw)
        assert info.converged
        xs.append(host(X))
        its.append(info.iterations)
        res = b - pb.rhs_from_solution(rp, ci, v, xs[-1])
        # the recursive norm meets 1e-9; the true one may differ by rounding
        assert np.abs(res).max() <= 2e-9 * np.abs(b).max()
    assert its[1] == its[0] and np.array_equal(xs[1], xs[0])
    # (other block sums in the inner products)
    assert abs(its[2] - its[0]) <= 1
