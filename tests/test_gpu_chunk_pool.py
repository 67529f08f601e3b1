"""Hierarchies on memory that earlier ones of the same handle gave back: the same
operators, cycles and solves bit for bit as on a fresh handle, larger and smaller
ones in turn, more alive at once than the pool has notes for, from several threads
and streams, after the handle's end; and the memory is back when the handle is gone."""
import gc
import threading

import numpy as np
import pytest
import torch

from linalglib_amd import lal, problems as pb
from oracle.oracle import CSR
from tests.gpu_util import DevCSR, dev, empty, host, log

pytestmark = pytest.mark.gpu


def _problem(n, seed):
    rng = np.random.default_rng(seed)
    rp, ci, v, m = pb.diffusion3d(n, cell_kappa=np.exp(rng.standard_normal((n, n, n))))
    return CSR(rp, ci, v, m, m), rng.uniform(-1, 1, m)


def _run(h, A, r):
    """(operators, one cycle, a solve) of a fresh hierarchy on h."""
    d = DevCSR(A)
    H = lal.Hierarchy(h, A.m, A.nnz, d.row_ptr, d.col_ind, d.val, build_f32=1)
    out = [a for l in range(H.levels + 1) for a in H.level(l, "A")[:3]]
    z = empty(A.m, torch.float64)
    H.precond(dev(r), z)
    X = torch.zeros(A.m, dtype=torch.float64, device="cuda")
    H.pcg_reliable(dev(r), X, rel_tol=1e-9, abs_tol=1e-300, max_iter=200)
    torch.cuda.synchronize()
    out += [host(z), host(X)]
    H.close()
    return out


def _same(a, b):
    return len(a) == len(b) and all(np.array_equal(x, y) for x, y in zip(a, b))


def test_reused_memory():
    probs = [_problem(n, n) for n in (20, 34, 9, 27)]
    fresh = [_run(lal.Handle(), *p) for p in probs]
    h = lal.Handle()
    for turn in range(3):
        for k in (1, 0, 3, 2, 1):
            log(f"reused memory: turn {turn}, problem {k}")
            assert _same(_run(h, *probs[k]), fresh[k])


def test_many_alive_and_the_handle_first():
    A, r = _problem(6, 1)
    h, d = lal.Handle(), DevCSR(A)
    hs = [lal.Hierarchy(h, A.m, A.nnz, d.row_ptr, d.col_ind, d.val) for _ in range(70)]
    ref = None
    for H in hs:  # (beyond 64 a hierarchy has a note of its own)
        X = torch.zeros(A.m, dtype=torch.float64, device="cuda")
        assert H.pcg(dev(r), X, rel_tol=1e-9, abs_tol=1e-300, max_iter=100).converged
        ref = host(X) if ref is None else ref
        assert np.array_equal(host(X), ref)
    h.close()
    for H in hs:
        H.close()


def test_threads_with_their_own_handles_and_streams():
    probs = [_problem(n, n) for n in (16, 22)]
    fresh = [_run(lal.Handle(), *p) for p in probs]
    bad = []

    def work(k):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                h = lal.Handle()
                for _ in range(4):
                    if not _same(_run(h, *probs[k]), fresh[k]):
                        bad.append(k)
        except Exception as e:  # noqa: BLE001 - reported below
            bad.append(repr(e))

    ts = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad


def test_memory_is_given_back():
    A, r = _problem(40, 3)
    _run(lal.Handle(), A, r)  # what the runtime itself keeps
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.mem_get_info()[0]
    h = lal.Handle()
    for _ in range(3):
        _run(h, A, r)
    h.close()
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # within the allocation granularity of a few small arrays
    assert before - torch.cuda.mem_get_info()[0] <= 8 << 20
