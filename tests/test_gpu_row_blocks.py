"""The device's row-block analysis: matrices whose rows end at, before and
after its tile (2048 rows) and block (256 rows, 256-2048 nonzeros) edges, rows
longer than a block, refused row pointers, and a hierarchy of more operators
than one launch takes."""
import numpy as np
import pytest
import torch

from linalglib_amd import lal, problems as pb
from oracle.oracle import CSR
from tests.gpu_util import DevCSR, dev, empty, host, log

pytestmark = pytest.mark.gpu


def _lengths(kind, m, rng):
    if kind == "short":
        return rng.integers(0, 6, m)
    if kind == "mixed":
        return np.where(rng.random(m) < 0.05, rng.integers(100, 400, m), rng.integers(0, 60, m))
    lens = np.full(m, 3)  # a row of several windows around a tile's edge
    for r in (0, 2046, 2047, 2048, m - 1):
        if r < m:
            lens[r] = 4500
    return lens


@pytest.mark.parametrize("kind", ["short", "mixed", "long"])
@pytest.mark.parametrize("m", [1, 255, 257, 2047, 2048, 2049, 6145])
def test_blocks_cover_every_row(m, kind):
    rng = np.random.default_rng(m)
    n = 7000
    lens = _lengths(kind, m, rng)
    rp = np.zeros(m + 1, np.int32)
    rp[1:] = np.cumsum(lens)
    ci = rng.integers(0, n, rp[-1]).astype(np.int32)
    v = rng.uniform(-1, 1, rp[-1])
    x = rng.uniform(-1, 1, n)
    log(f"row blocks m={m} {kind}")
    h = lal.Handle()
    d = DevCSR(CSR(rp, ci, v, m, n))
    X = dev(x)
    rows = np.repeat(np.arange(m), lens)
    ref = np.zeros(m, np.longdouble)
    np.add.at(ref, rows, v.astype(np.longdouble) * x[ci])
    # products and sums in any order: (len + 3) u sum |a x| (recursive summation)
    tol = (lens + 3) * 2.0 ** -53 * np.bincount(rows, weights=np.abs(v * x[ci]), minlength=m)
    for exact in (False, True):
        desc = lal.CsrDescr(h, m, n, int(rp[-1]), d.row_ptr, d.col_ind, exact=exact)
        y = torch.full((m,), np.nan, dtype=torch.float64, device="cuda")
        lal.call("lal_csrmv_f64", h.h, desc.d, m, n, int(rp[-1]), 1.0, lal.ptr(d.row_ptr),
                 lal.ptr(d.col_ind), lal.ptr(d.val), lal.ptr(X), 0.0, lal.ptr(y))
        assert np.all(np.abs(host(y) - ref) <= tol)


def test_refused_patterns():
    h = lal.Handle()
    m, n = 5000, 40
    rp = np.arange(m + 1, dtype=np.int32)
    ci = np.zeros(m, np.int32)

    def analyse(rp, ci, m, nnz):
        a, b = dev(rp, np.int32), dev(ci, np.int32)
        return lal.CsrDescr(h, m, n, nnz, a, b)

    for at, to in ((0, 1), (m, m - 1), (2048, 100), (4999, -3), (1, 2 ** 31 - 1)):
        bad = rp.copy()
        bad[at] = to
        log(f"refused row_ptr[{at}] = {to}")
        with pytest.raises(lal.LalError) as e:
            analyse(bad, ci, m, m)
        assert e.value.status == 1
    for at, to in ((0, n), (m - 1, -1)):
        bad = ci.copy()
        bad[at] = to
        with pytest.raises(lal.LalError) as e:
            analyse(rp, bad, m, m)
        assert e.value.status == 1
    with pytest.raises(lal.LalError):
        analyse(np.array([3], np.int32), ci[:1], 0, 0)
    analyse(np.array([0], np.int32), ci[:1], 0, 0)  # no rows: fine
    analyse(rp, ci, m, m)  # and the flags of the refused ones are gone


def test_hierarchy_of_more_operators_than_a_launch(oracle):
    """A chain coarsens by about three per level: 9 levels and more, over 24
    operators.  Every one is analysed (a fast V-cycle agrees with the
    oracle's, tolerance as for the other fast V-cycles) and keeps 16-bit
    columns, as its blocks span few."""
    rp, ci, v, m = pb.poisson2d(60011, 1)
    h = lal.Handle()
    d = DevCSR(CSR(rp, ci, v, m, m))
    H = lal.Hierarchy(h, m, len(ci), d.row_ptr, d.col_ind, d.val)
    log(f"chain hierarchy of {H.levels} levels")
    assert 3 * H.levels > 24
    for lvl in range(H.levels):
        assert all(H.column_bytes(lvl, k) == 2 for k in "APR")
    r = np.random.default_rng(4).uniform(-1, 1, m)
    z = empty(m, torch.float64)
    H.precond(dev(r), z, 1, 1)
    ref = oracle.saamg_setup(CSR(rp, ci, v, m, m)).precond(r, 1, 1, 1)
    assert np.linalg.norm(host(z) - ref) <= 1e-10 * np.linalg.norm(ref)
