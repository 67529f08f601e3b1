"""The column lists' code on the host: every entry that the list kernel gathers,
the padding of an odd list included, is a column of the block and below the
matrix's column count, for blocks with and without offsets of 65536 and more in
one matrix (the restriction of a grid with long lines) and at the lists' ends."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from linalglib_amd import problems as pb
from oracle.oracle import CSR

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("lists") / "list_columns.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC",
                    "-I" + os.path.join(ROOT, "linalglib_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "list_columns.cpp"), "-o", so], check=True)
    return C.CDLL(so)


def _gathered(code, cols):
    """(stored offsets, decoded columns) of a block's list, padding included."""
    distinct = np.unique(cols)
    off = distinct - distinct[0]
    near = int((off < 65536).sum())
    split = code.lists_split(len(off), near)
    assert 0 <= split < 4096  # its field in the block's word
    stored = (off & 0xffff).astype(np.uint16)
    if len(stored) & 1:
        stored = np.append(stored, stored[-1])
    got = np.empty(len(stored), np.int32)
    code.lists_decode(stored.ctypes.data_as(C.c_void_p), len(stored), int(distinct[0]), split,
                      got.ctypes.data_as(C.c_void_p))
    assert np.array_equal(got[:len(distinct)], distinct)
    return got


@pytest.mark.parametrize("far", [0, 1, 2, 5])
@pytest.mark.parametrize("near", [1, 2, 3, 2039])
def test_ends_of_a_list(code, near, far):
    # a block whose last columns are the matrix's
    cols = np.concatenate([1000 + np.arange(near), 1000 + 65536 + 7 * np.arange(far)])
    got = _gathered(code, cols)
    assert got.max() == cols.max()


def _blocks(rp, rows_per_tile=2048, rows=256, cap=2044):
    """Row blocks as the analysis packs them."""
    m = len(rp) - 1
    while cap > 256 and rp[-1] // 256 < cap:
        cap >>= 1
    for t in range(0, m, rows_per_tile):
        end, r = min(m, t + rows_per_tile), t
        while r < end:
            e = r + 1
            while e < end and e - r < rows and rp[e + 1] - rp[r] <= cap:
                e += 1
            yield r, e
            r = e


@pytest.mark.parametrize("nx,ny", [(15001, 9), (20011, 8)])
def test_restriction_of_long_lines(code, oracle, nx, ny):
    rp, ci, v, m = pb.poisson2d(nx, ny)
    R = oracle.saamg_setup(CSR(rp, ci, v, m, m)).get(0, "R")
    spans, odd_near = [], 0
    for r0, r1 in _blocks(R.row_ptr):
        cols = R.col_ind[R.row_ptr[r0]:R.row_ptr[r1]]
        got = _gathered(code, cols)
        assert got.max() == cols.max() < m
        spans.append(int(cols.max()) - int(cols.min()))
        odd_near += spans[-1] < 65536 and len(np.unique(cols)) & 1
    assert 65535 < max(spans) < 131072 and odd_near > 0  # both kinds of block are there
