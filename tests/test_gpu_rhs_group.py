"""The FP64 lane-group form of the rhs! kernel (csrc/rhs_group_kernel.hpp) and
its logarithm-free means, where they can go wrong: element counts below and not
a multiple of the tile (1, 8, 960 with mortars), and states whose neighbouring
nodes differ by up to a factor of twenty in some lines only, so that waves mix
pairs of the series and of the logarithm; against the FP64 oracle, du within
the FP64 parity bound (1e-12 of its largest value) and one Runge-Kutta stage
through it."""
import os

import numpy as np
import pytest

from cases import Case, oracle_cfg, oracle_mesh, product_semi

pytestmark = pytest.mark.gpu

BOX = (((-1.0,) * 3, (1.0,) * 3),)
CASES = [
    Case("euler3d_one_element", 3, "euler", 0, "fd", "ranocha"),
    Case("euler3d_ranocha_llf", 3, "euler", 2, "fd", "ranocha"),
    Case("euler3d_ranocha_ec", 3, "euler", 1, "fd", "ranocha", "ranocha"),
    Case("euler3d_shima_llf_naive", 3, "euler", 1, "fd", "shima_etal", "llf_naive"),
    Case("euler3d_ranocha_llf_p1", 3, "euler", 2, "fd", "ranocha", polydeg=1),
    Case("euler3d_hg", 3, "euler", 1, "hg", "ranocha", "ranocha", "ranocha", alpha_min=0.0),
    Case("euler3d_mortars", 3, "euler", 3, "fd", "ranocha", patches=BOX),
    Case("euler2d_ranocha_llf", 2, "euler", 2, "fd", "ranocha"),
    Case("euler2d_hg", 2, "euler", 3, "hg", "ranocha", alpha_min=0.0),
    Case("mhd3d", 3, "mhd", 1, "fd", "hindenlang_gassner", gamma=5 / 3),
    Case("mhd3d_ec", 3, "mhd", 0, "fd", "hindenlang_gassner", "hindenlang_gassner", gamma=5 / 3),
    Case("mhd2d_hg", 2, "mhd", 2, "hg", "hindenlang_gassner", "hindenlang_gassner", "hindenlang_gassner", gamma=1.4,
         alpha_min=0.0),
]


def _jumps(case, mesh):
    """Smooth-ish random primitives, with one node in twenty off by a factor
    of up to twenty in density and pressure (on the mortar mesh one element in
    twenty: a face with such nodes interpolates to negative pressures there,
    where the oracle itself is NaN)."""
    rng = np.random.default_rng(7)
    shape = (mesh.nelements,) + (case.polydeg + 1,) * case.ndims
    rho, p = 1.0 + 0.05 * rng.random(shape), 1.0 + 0.05 * rng.random(shape)
    where = shape if not case.patches else (mesh.nelements,) + (1,) * case.ndims
    for q in (rho, p):
        q *= np.where(rng.random(where) < 0.05, 20.0 ** rng.uniform(-1.0, 1.0, where), 1.0)
    nvel = 3 if case.equation == "mhd" else case.ndims
    v = [0.2 * rng.standard_normal(shape) for _ in range(nvel)]
    en = p / (case.gamma - 1.0) + 0.5 * rho * sum(x * x for x in v)
    if case.equation == "mhd":
        B = [0.3 * rng.standard_normal(shape) for _ in range(3)]
        psi = 0.1 * rng.standard_normal(shape)
        en = en + 0.5 * sum(x * x for x in B) + 0.5 * psi * psi
        return np.ascontiguousarray(np.stack([rho] + [rho * x for x in v] + [en] + B + [psi], -1))
    return np.ascontiguousarray(np.stack([rho] + [rho * x for x in v] + [en], -1))


@pytest.mark.parametrize("np_form", [False, True], ids=["group", "node_parallel"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: c.name)
def test_rhs_with_jumps(th, oracle, case, np_form, monkeypatch):
    import torch
    monkeypatch.setenv("TRIXI_HIP_NP_LANES", str(1 << 40) if np_form else "0")
    mesh = oracle_mesh(oracle, case)
    u = _jumps(case, mesh)
    ref = oracle.rhs(oracle_cfg(oracle, case), mesh, u)
    semi = product_semi(th, case, "fp64")
    try:
        ud = th.pack(torch.from_numpy(u).cuda(), semi)
        du = torch.empty_like(ud)
        th.rhs_hip_(du, ud, semi, 0.0)
        got = th.wrap_array_native(du, semi).cpu().numpy()
        err = np.abs(got - ref).max() / np.abs(ref).max()
        print(f"{case.name}: {err:.3e}", flush=True)
        assert err <= 1e-12
        dt = 1e-4
        k = torch.zeros_like(ud)
        uo = torch.empty_like(ud)
        th.rk_stage(ud, k, uo, 0, 0.0, dt, semi)
        ks = th.wrap_array_native(k, semi).cpu().numpy()
        assert np.abs(ks - dt * ref).max() <= 1e-12 * dt * np.abs(ref).max()
    finally:
        semi.close()
