"""What a context keeps of destroyed hierarchies goes back to the driver before an
allocation of the library fails, whichever context keeps it and whichever call
allocates; all contexts together keep at most 1/32 of the device's memory, and
nothing large while the device is short of it."""
import ctypes as C
import gc

import numpy as np
import pytest
import torch

from linalglib_amd import lal, problems as pb
from oracle.oracle import CSR
from tests.gpu_util import DevCSR, empty, log

pytestmark = pytest.mark.gpu

GB = 1 << 30


def _free():
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0]


def _fill(leave):
    """Tensors that take the device's memory but for about `leave` bytes."""
    held = []
    while _free() > leave + (64 << 20):
        held.append(torch.empty(min(_free() - leave, 32 * GB), dtype=torch.uint8, device="cuda"))
    return held


@pytest.fixture(scope="module")
def grid():
    rp, ci, v, m = pb.poisson3d(96)
    return DevCSR(CSR(rp, ci, v, m, m))


def _hierarchy(h, d):
    return lal.Hierarchy(h, d.m, d.nnz, d.row_ptr, d.col_ind, d.val, build_f32=1)


def _pooled(h, d):
    """Builds and destroys a hierarchy on h; the bytes the pool keeps of it."""
    _hierarchy(h, d).close()  # (the runtime's own growth)
    h.close()
    before = _free()
    h = lal.Handle()
    _hierarchy(h, d).close()
    return h, before - _free()


@pytest.mark.parametrize("call", ["alloc", "transpose", "hierarchy"])
def test_a_failing_allocation_empties_the_pools(grid, call):
    h, kept = _pooled(lal.Handle(), grid)
    assert kept > 0.8 * GB  # else the case shows nothing
    other = lal.Handle()
    if call == "transpose":
        # one integer per entry of scratch, beside operands that are there
        nnz, n = 180 << 20, 1 << 24
        rp = torch.arange(0, nnz + 1, 16, dtype=torch.int32, device="cuda")
        ci = torch.arange(nnz, dtype=torch.int32, device="cuda") & (n - 1)
        v = torch.ones(nnz, dtype=torch.float32, device="cuda")
        trp, tci, tv = empty(n + 1, torch.int32), torch.empty_like(ci), torch.empty_like(v)
    held = _fill(GB // 2)
    room = _free()
    log(f"memory pressure {call}: {kept >> 20} MB kept, {room >> 20} MB free")
    assert room < 0.6 * GB
    if call == "alloc":
        p = C.c_void_p()
        lal.call("lal_alloc", C.byref(p), room + (256 << 20))
        lal.call("lal_free", p)
    elif call == "transpose":
        assert 4 * nnz > room
        lal.call("lal_transpose_f32", other.h, nnz // 16, n, nnz, lal.ptr(rp), lal.ptr(ci), lal.ptr(v),
                 lal.ptr(trp), lal.ptr(tci), lal.ptr(tv))
        torch.cuda.synchronize()
        assert int(trp[-1]) == nnz and int(tci[-1]) == (nnz // n * n - 1) // 16
    else:
        _hierarchy(other, grid).close()
    del held
    for q in (h, other):
        q.close()


def test_all_contexts_share_one_bound(grid):
    handles = [lal.Handle() for _ in range(12)]
    h, kept = _pooled(lal.Handle(), grid)
    h.close()
    before, total = _free(), torch.cuda.mem_get_info()[1]
    assert kept * len(handles) > total // 32  # else the case shows nothing
    for q in handles:
        _hierarchy(q, grid).close()
    # and the allocation granularity of a few small arrays
    assert before - _free() <= total // 32 + (64 << 20)
    for q in handles:
        q.close()


def test_nothing_is_kept_while_memory_is_short(grid):
    h = lal.Handle()
    total = torch.cuda.mem_get_info()[1]
    held = _fill(total // 16)
    before = _free()
    _hierarchy(h, grid).close()
    assert before - _free() <= 32 << 20
    del held
    h.close()


def test_a_build_short_of_memory_does_without_the_extras():
    """128^3: 2.1 GB with Q, the column lists and the dense cycle operator, 1.1
    without them: the same operators, a V-cycle within the fast ones' bar, and a
    solve."""
    rp, ci, v, m = pb.poisson3d(128)
    d = DevCSR(CSR(rp, ci, v, m, m))
    h = lal.Handle()
    r = torch.from_numpy(np.random.default_rng(3).uniform(-1, 1, m)).cuda()
    z, zl, x = empty(m, torch.float64), empty(m, torch.float64), empty(m, torch.float64)

    def build():
        return lal.Hierarchy(h, m, d.nnz, d.row_ptr, d.col_ind, d.val)

    H = build()
    H.precond(r, z)
    ops = [H.level(l, k)[:3] for l in (1, 3) for k in "APR" if l < H.levels]
    H.close()
    h.close()
    h = lal.Handle()
    held = _fill(1500 << 20)
    before = _free()
    log(f"build with {before >> 20} MB free")
    H = build()
    assert before - _free() < 1200 << 20
    H.precond(r, zl)
    info = H.pcg(r, x, rel_tol=1e-8, abs_tol=1e-300, max_iter=100)
    assert info.converged
    lean = [H.level(l, k)[:3] for l in (1, 3) for k in "APR" if l < H.levels]
    assert all(np.array_equal(a, b) for o, p in zip(ops, lean) for a, b in zip(o, p))
    assert float((zl - z).norm()) <= 1e-10 * float(z.norm())
    del held
    H.close()
    h.close()
