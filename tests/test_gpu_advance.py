"""The native time loop (trixi_hip_advance) against the loop of single steps:
the same times, step counts and states, bit for bit, for CFL and fixed steps,
runs that end on the final time or on maxiters, within and beyond one chunk of
queued steps, with analysis in between, and the refused arguments."""
import ctypes

import pytest

from cases import Case, product_semi

pytestmark = pytest.mark.gpu

CASES = [
    (Case("advection2d", 2, "linadv", 2, ic="convergence_test", cmin=-1.0, cmax=1.0), "fp64"),
    (Case("euler2d_hg", 2, "euler", 3, "hg", "ranocha", ic="weak_blast_wave_seeded"), "fp64"),
    (Case("euler3d_level5", 3, "euler", 4, "fd", "ranocha", ic="smooth_periodic"), "fp64"),
    (Case("euler3d_mixed", 3, "euler", 2, "fd", "ranocha", ic="smooth_periodic"), "mixed"),
    (Case("euler3d_fp32", 3, "euler", 2, "fd", "ranocha", ic="smooth_periodic"), "fp32"),
    (Case("euler2d_source_dirichlet", 2, "euler", 2, cmin=0.0, cmax=2.0, ic="convergence_test", periodic=False,
          bc_state="convergence_test", source="convergence_test"), "fp64"),
    (Case("advection3d_mortar", 3, "linadv", 2, cmin=-1.0, cmax=1.0, ic="convergence_test", advection=(0.2, -0.7, 0.5),
          patches=(((0.0, -1.0, -1.0), (1.0, 1.0, 1.0)),)), "fp64"),
]


@pytest.mark.parametrize("end", ["t_end", "maxiters", "long", "none", "dt", "analysis"])
@pytest.mark.parametrize("case,precision", CASES, ids=lambda x: getattr(x, "name", x))
def test_advance_equals_single_steps(th, case, precision, end):
    import torch

    class OwnStepsize(th.StepsizeCallback):  # not the built class: solve() takes single steps
        pass

    semi = product_semi(th, case, precision)
    try:
        h = 0.4 * th.max_dt(th.compute_coefficients(0.0, semi), semi)
        t1 = {"t_end": 3.3 * h, "maxiters": 1e3, "long": 1e3, "none": 0.0, "dt": 2.5 * h, "analysis": 6.2 * h}[end]
        iters = {"maxiters": 5, "long": 70}.get(end, 10 ** 6)
        ode = th.semidiscretizeHIP(semi, (0.0, t1))
        out = []
        for cls in (th.StepsizeCallback, OwnStepsize):
            cb = [] if end == "dt" else [cls(0.4)]
            if end == "analysis":
                if semi.fp32_state or case.ic not in ("convergence_test", "smooth_periodic"):
                    pytest.skip("no error norms of this state")
                cb.append(th.AnalysisCallback(semi, interval=4))
            if end == "dt" and cls is OwnStepsize:
                # single steps through rk_step
                u, k, t, n = ode.u0.clone(), torch.zeros_like(ode.u0), 0.0, 0
                st = torch.cuda.Stream()
                st.wait_stream(torch.cuda.current_stream())
                while t < t1:
                    step = min(h, t1 - t)
                    step, t = (t1 - t, t1) if t + h >= t1 else (h, t + h)
                    th.rk_step(u, k, t - step if t != t1 else t1 - step, step, semi, stream=st)
                    n += 1
                st.synchronize()
                out.append((u, t, n, []))
                continue
            sol = th.solve(ode, th.CarpenterKennedy2N54(), dt=h if end == "dt" else None, callback=cb, maxiters=iters)
            out.append((sol.u, sol.t, sol.nsteps, cb[1].history if end == "analysis" else []))
        (ua, ta, na, ha), (ub, tb, nb, hb) = out
        assert (ta, na) == (tb, nb)
        if not (end == "dt" and case.source):  # (that loop's stage times may differ in the last bit)
            assert torch.equal(ua, ub)
        else:
            assert torch.allclose(ua, ub, rtol=1e-13, atol=1e-14)
        assert [x[0] for x in ha] == [x[0] for x in hb]
        assert all((p == q).all() for x, y in zip(ha, hb) for p, q in zip(x[1:], y[1:]))
    finally:
        semi.close()


def test_advance_refuses(th):
    import torch
    semi = product_semi(th, CASES[0][0], "fp64")
    try:
        u = th.compute_coefficients(0.0, semi)
        k = torch.zeros_like(u)
        n, t = ctypes.c_int64(), ctypes.c_double(0.0)
        lib, p = th._lib.lib(), lambda x: ctypes.c_void_p(x.data_ptr())
        args = (ctypes.byref(t), 1.0, 0.5, 0.0, 3, ctypes.byref(n), None)
        assert lib.trixi_hip_advance(semi.ctx, p(u), p(u), *args) == th._lib.EINVAL
        assert lib.trixi_hip_advance(semi.ctx, None, p(k), *args) == th._lib.EINVAL
        assert lib.trixi_hip_advance_f32(semi.ctx, p(u), p(k), *args) == th._lib.EINVAL
        assert lib.trixi_hip_advance(semi.ctx, p(u), p(k), ctypes.byref(t), 1.0, 0.0, 0.0, 3, ctypes.byref(n),
                                     None) == th._lib.EINVAL
    finally:
        semi.close()
