"""PCG's reductions inside its products: inner products as one partial per row
block (one block, around the 512 partials of the separate kernels, more blocks
than the fused ones take), the norm finished by the cycle's first kernel, with
replayed graphs and without, and the paths that keep separate kernels (two
post-sweeps, other smoothers, a caller's unaligned operator)."""
import numpy as np
import pytest
import torch

from linalglib_amd import lal, problems as pb
from oracle.oracle import CSR
from tests.gpu_util import DevCSR, dev, host, log

pytestmark = pytest.mark.gpu

SIZES = {
    "one_block": lambda: pb.poisson2d(9, 7),
    "blocks_512": lambda: pb.poisson2d(360, 362),   # about 510 blocks of 256 rows
    "graph_limit": lambda: pb.poisson2d(256, 256),  # replayed as a graph
    "beyond_graph": lambda: pb.poisson2d(257, 256),
    "rows_262144": lambda: pb.poisson2d(512, 512),
    "beyond_parts": lambda: pb.poisson3d(102),      # 4146 blocks of 256 rows
}


def _solve(H, b, m, solve="pcg", **kw):
    X = torch.zeros(m, dtype=torch.float64, device="cuda")
    info = getattr(H, solve)(dev(b), X, rel_tol=1e-9, abs_tol=1e-300, max_iter=300, **kw)
    return host(X), info


@pytest.mark.parametrize("name", sorted(SIZES))
def test_pcg_reductions(name):
    rp, ci, v, m = SIZES[name]()
    log(f"PCG reductions {name}")
    h = lal.Handle()
    d = DevCSR(CSR(rp, ci, v, m, m))
    H = lal.Hierarchy(h, m, len(ci), d.row_ptr, d.col_ind, d.val, build_f32=1)
    E = lal.Hierarchy(h, m, len(ci), d.row_ptr, d.col_ind, d.val, exact=1)
    b = pb.rhs_from_solution(rp, ci, v, np.random.default_rng(6).uniform(-1, 1, m))
    _, ref = _solve(E, b, m)
    for solve in ("pcg", "pcg_mixed", "pcg_reliable"):
        first = None
        for _ in range(3):  # eager, captured, replayed
            x, info = _solve(H, b, m, solve)
            assert info.converged
            # the same recurrences as the separate kernels', up to rounding
            # (FP32 levels, FP32 vectors: a few steps more)
            assert info.iterations <= ref.iterations + (1 if solve == "pcg" else 5)
            res = b - pb.rhs_from_solution(rp, ci, v, x)
            assert np.abs(res).max() <= 2e-9 * np.abs(b).max()
            first = x if first is None else first
            assert np.array_equal(x, first)
    x, info = _solve(H, b, m, n2=2)
    assert info.converged
    if m < 1000:
        x, info = _solve(H, b, m, smoother=4)  # SSOR: symmetric
        assert info.converged
    b[m // 2] = np.nan
    for solve in ("pcg", "pcg_mixed", "pcg_reliable"):
        _, info = _solve(H, b, m, solve)
        assert not info.converged
