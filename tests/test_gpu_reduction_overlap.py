"""Reductions that run at the same time on one GPU.  Contexts have buffers of
their own, so their reductions are independent.  trixi_hip_max_dt_noalloc shares
its partials between contexts: the results of calls that overlap are undefined,
but every later call is right again."""
import ctypes
import threading

import numpy as np
import pytest

from cases import Case, product_semi

pytestmark = pytest.mark.gpu

CALLS = 150  # per thread


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.fixture()
def contexts(th, torch):
    # grids of 1, 4 and 256 blocks (16 elements a block)
    out = []
    for nd, level, scale in ((2, 2, 1.0), (3, 2, 2.0), (3, 4, 3.0)):
        semi = product_semi(th, Case("overlap", nd, "euler", level, "fd", "ranocha", ic="smooth_periodic"))
        u = th.compute_coefficients(0.0, semi)
        u.view(semi.nvariables, -1)[1:1 + nd].mul_(scale)
        out.append((semi, u))
    torch.cuda.synchronize()
    yield out
    for semi, _ in out:
        semi.close()


def _in_threads(torch, contexts, work):
    """work(semi, u, stream) CALLS times per context, a thread and a stream each."""
    errors, start = [], threading.Barrier(len(contexts))

    def run(semi, u):
        try:
            stream = torch.cuda.Stream()
            start.wait()
            for _ in range(CALLS):
                work(semi, u, ctypes.c_void_p(stream.cuda_stream))
        except BaseException as e:
            errors.append(e)

    threads = [threading.Thread(target=run, args=c) for c in contexts]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if errors:
        raise errors[0]


def _max_dt(th, name, semi, u, stream):
    out = ctypes.c_double()
    th._lib.check(getattr(th._lib.lib(), name)(semi.ctx, ctypes.c_void_p(u.data_ptr()), ctypes.byref(out), stream))
    return out.value


def test_noalloc_is_right_again_after_an_overlap(th, torch, contexts):
    ref = [th.max_dt(u, semi) for semi, u in contexts]
    _in_threads(torch, contexts, lambda semi, u, s: _max_dt(th, "trixi_hip_max_dt_noalloc", semi, u, s))
    torch.cuda.synchronize()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        for (semi, u), r in zip(contexts, ref):
            assert _max_dt(th, "trixi_hip_max_dt_noalloc", semi, u, stream) == r
            assert th.max_dt(u, semi) == r


def test_contexts_reduce_independently(th, torch, contexts):
    want = {}
    for semi, u in contexts:
        want[semi] = (th.max_dt(u, semi), th.integrate(u, semi), th.calc_error_norms(u, 0.3, semi))
    torch.cuda.synchronize()

    def work(semi, u, s):
        dt, integrals, (l2, linf) = want[semi]
        assert _max_dt(th, "trixi_hip_max_dt", semi, u, s) == dt
        lib, p = th._lib.lib(), ctypes.c_void_p(u.data_ptr())
        out, e2, einf = (np.zeros(semi.nvariables) for _ in range(3))
        ptr = lambda x: x.ctypes.data_as(ctypes.c_void_p)
        th._lib.check(lib.trixi_hip_integrate(semi.ctx, p, ptr(out), s))
        ic = semi.initial_condition
        th._lib.check(lib.trixi_hip_error_norms(semi.ctx, p, ic.ic_id, 0.3, ic.seed, ptr(e2), ptr(einf), s))
        assert np.array_equal(out, integrals) and np.array_equal(e2, l2) and np.array_equal(einf, linf)

    _in_threads(torch, contexts, work)
