"""The FP64 lane-group form of the adjoint (csrc/vjp_group_kernel.hpp) where it
can go wrong: element counts below and at the tile, remainders of it, boundary
faces, and states whose neighbouring nodes differ by up to a factor of twenty in
some lines only, so that waves mix pairs of the series and of the logarithm;
J^T vbar with J column by column from the oracle's dual numbers, within the
bound of the adjoint's other tests (1e-11 of the largest value), and the
accumulation into ubar.  The fused reverse Runge-Kutta stage against the
direction-group form of the same step, within the same bound."""
import numpy as np
import pytest

from cases import Case, oracle_cfg, oracle_mesh, product_semi
from test_gpu_rhs_group import _jumps

pytestmark = pytest.mark.gpu

OPEN = dict(cmin=0.0, cmax=2.0, periodic=False, bc_state="convergence_test", t=0.3)
CASES = [
    Case("euler3d_one_element", 3, "euler", 0, "fd", "ranocha"),
    Case("euler3d_ranocha_llf", 3, "euler", 1, "fd", "ranocha"),
    Case("euler3d_ranocha_ec", 3, "euler", 0, "fd", "ranocha", "ranocha"),
    Case("euler3d_shima_llf_naive", 3, "euler", 1, "fd", "shima_etal", "llf_naive"),
    Case("euler3d_dirichlet", 3, "euler", 0, "fd", "ranocha", **OPEN),
    Case("euler2d_one_element", 2, "euler", 0, "fd", "ranocha"),
    Case("euler2d_ranocha_llf", 2, "euler", 2, "fd", "ranocha"),
    Case("euler2d_ranocha_llf_naive", 2, "euler", 3, "fd", "ranocha", "llf_naive"),
    Case("euler2d_shima_ec", 2, "euler", 1, "fd", "shima_etal", "shima_etal"),
    Case("euler2d_dirichlet", 2, "euler", 2, "fd", "ranocha", **OPEN),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: c.name)
def test_vjp_with_jumps(th, oracle, case, monkeypatch):
    import torch
    O = oracle
    monkeypatch.setenv("TRIXI_HIP_VJP_PD_LANES", "0")
    cfg, mesh = oracle_cfg(O, case), oracle_mesh(O, case)
    u = _jumps(case, mesh)
    semi = product_semi(th, case)
    J = O.jacobian(cfg, mesh, u, case.t)
    vbar = np.random.default_rng(3).standard_normal(u.shape)
    expect = (J.T @ vbar.ravel()).reshape(u.shape)
    ud, vd = (th.pack(torch.from_numpy(x).cuda(), semi) for x in (u, vbar))
    ubar = torch.empty_like(ud)
    th.rhs_vjp(ubar, ud, vd, semi, t=case.t)
    th.rhs_vjp(ubar, ud, vd, semi, t=case.t, alpha=3.0, beta=2.0)
    got = th.wrap_array_native(ubar, semi).cpu().numpy()
    assert np.abs(got - 5 * expect).max() < 1e-11 * np.abs(expect).max()
    semi.close()


@pytest.mark.parametrize("case", CASES[1:2] + CASES[6:7], ids=lambda c: c.name)
def test_reverse_step(th, oracle, case, monkeypatch):
    import torch
    u = _jumps(case, oracle_mesh(oracle, case))
    vbar = np.random.default_rng(4).standard_normal(u.shape)
    out = []
    for lanes in ("0", "1000000"):
        monkeypatch.setenv("TRIXI_HIP_VJP_PD_LANES", lanes)
        semi = product_semi(th, case)
        th.enable_adjoint(semi)
        ud, ubar = (th.pack(torch.from_numpy(x).cuda(), semi) for x in (u, vbar))
        th.rk_step_vjp(ud, ubar, 0.0, 1e-4, semi)
        out.append(th.wrap_array_native(ubar, semi).cpu().numpy())
        semi.close()
    assert np.abs(out[0] - out[1]).max() < 1e-11 * np.abs(out[1]).max()
