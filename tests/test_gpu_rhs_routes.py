"""The kernels that one rhs! configuration takes by mesh size: on large meshes rhs!
in 2D and of some 3D shock capturing runs the line form and the Runge-Kutta stages
lane groups (csrc/launch_rhs.hpp), so the first stage of a step of size one (k =
rhs!) compares the two over the forms built; and lane groups on meshes whose element count
leaves a partial tile after full ones, which refined meshes have, against the oracle."""
import numpy as np
import pytest

from cases import Case, oracle_cfg, oracle_mesh, product_semi
from test_gpu_rhs_group import _jumps

pytestmark = pytest.mark.gpu

HG = "hindenlang_gassner"
LARGE = (
    [Case(f"euler2d_{v}_{s}", 2, "euler", 7, "fd", v, s) for v in ("ranocha", "shima_etal") for s in ("llf", "llf_naive", v)]
    + [Case(f"euler2d_hg_{v}_{s}", 2, "euler", 7, "hg", v, s, s, alpha_min=0.0)
       for v in ("ranocha", "shima_etal") for s in ("llf", "llf_naive")]
    + [Case(f"mhd2d_{v}_{s}", 2, "mhd", 7, "fd", v, s, gamma=5 / 3)
       for v, s in ((HG, "llf"), (HG, "llf_naive"), (HG, HG), (HG, "hlle"), ("central", "llf"))]
    + [Case(f"mhd2d_hg_{s}", 2, "mhd", 7, "hg", HG, s, s, gamma=5 / 3, alpha_min=0.0) for s in ("llf", HG)]
    + [Case(f"euler3d_hg_{v}_{s}", 3, "euler", 4, "hg", v, s, s, alpha_min=0.0)
       for v, s in (("ranocha", "llf"), ("ranocha", "llf_naive"), ("ranocha", "ranocha"), ("shima_etal", "llf"),
                    ("shima_etal", "llf_naive"))])


@pytest.mark.parametrize("case", LARGE, ids=lambda c: c.name)
def test_large_mesh_rhs_equals_first_stage(th, oracle, case):
    import torch
    u = _jumps(case, oracle_mesh(oracle, case))
    semi = product_semi(th, case)
    try:
        ud = th.pack(torch.from_numpy(u).cuda(), semi)
        du, k, uo = torch.empty_like(ud), torch.zeros_like(ud), torch.empty_like(ud)
        th.rhs_hip_(du, ud, semi, 0.0)
        th.rk_stage(ud, k, uo, 0, 0.0, 1.0, semi)
        # both within the parity bound of the exact sums
        err = float((du - k).abs().max() / du.abs().max())
        print(f"{case.name}: {err:.3e}", flush=True)
        assert err <= 2e-12
    finally:
        semi.close()


ONE_3D, ONE_2D = (((-2.0,) * 3, (0.0,) * 3),), (((-2.0, -2.0), (-1.5, -1.5)),)
PARTIAL = [
    (15, Case("euler3d_fd", 3, "euler", 1, "fd", "ranocha", patches=ONE_3D)),
    (15, Case("euler3d_hg", 3, "euler", 1, "hg", "ranocha", alpha_min=0.0, patches=ONE_3D)),
    (15, Case("mhd3d", 3, "mhd", 1, "fd", HG, gamma=5 / 3, patches=ONE_3D)),
    (67, Case("euler2d_fd", 2, "euler", 3, "fd", "ranocha", patches=ONE_2D)),
    (67, Case("euler2d_hg", 2, "euler", 3, "hg", "ranocha", alpha_min=0.0, patches=ONE_2D)),
    (67, Case("mhd2d", 2, "mhd", 3, "fd", HG, "hlle", gamma=5 / 3, patches=ONE_2D)),
]


@pytest.mark.parametrize("elements,case", PARTIAL, ids=lambda x: x.name if isinstance(x, Case) else str(x))
def test_partial_tile(th, oracle, elements, case):
    import torch
    mesh = oracle_mesh(oracle, case)
    assert mesh.nelements == elements
    u = _jumps(case, mesh)
    ref = oracle.rhs(oracle_cfg(oracle, case), mesh, u)
    semi = product_semi(th, case)
    try:
        ud = th.pack(torch.from_numpy(u).cuda(), semi)
        # vectors that end in the middle of a longer buffer: nothing may be written past them
        guard = 4096
        whole = [torch.full((ud.numel() + guard,), 7.0, dtype=torch.float64, device="cuda") for _ in range(3)]
        du, k, uo = (w[:ud.numel()] for w in whole)
        th.rhs_hip_(du, ud, semi, 0.0)
        got = th.wrap_array_native(du, semi).cpu().numpy()
        assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
        # a stage that reads its register: k <- A k + dt rhs, u_out = u + B k
        A, B = oracle.ck2n54_coefficients()[:2]
        dt, k0 = 1e-4, np.random.default_rng(5).standard_normal(u.shape) * 1e-4
        k.copy_(th.pack(torch.from_numpy(k0).cuda(), semi))
        th.rk_stage(ud, k, uo, 2, 0.0, dt, semi)
        want = A[2] * k0 + dt * ref
        ks = th.wrap_array_native(k, semi).cpu().numpy()
        assert np.abs(ks - want).max() <= 1e-12 * dt * np.abs(ref).max() + 1e-15 * np.abs(k0).max()
        us = th.wrap_array_native(uo, semi).cpu().numpy()
        assert np.abs(us - (u + B[2] * ks)).max() <= 4e-16 * np.abs(u).max()
        assert all(bool((w[ud.numel():] == 7.0).all()) for w in whole)
    finally:
        semi.close()
