"""States a run has broken: one node not a number, with nonpositive or zero density or
pressure, or infinite.  The FP64 rhs! must be a number wherever the oracle's is, and
not elsewhere (how far such a node reaches: the lines through it and its face
neighbours), in lane groups and in the node-parallel form.  And max_dt of an FP32
state is that of the widened state."""
import numpy as np
import pytest

from cases import Case, oracle_cfg, oracle_mesh, product_semi

pytestmark = pytest.mark.gpu

HG = "hindenlang_gassner"
CASES = [Case("euler3d", 3, "euler", 2, "fd", "ranocha"), Case("euler3d_ec", 3, "euler", 2, "fd", "ranocha", "ranocha"),
         Case("euler3d_shima", 3, "euler", 2, "fd", "shima_etal"), Case("euler2d_hg", 2, "euler", 3, "hg", "ranocha"),
         Case("mhd3d", 3, "mhd", 1, "fd", HG), Case("mhd3d_hlle", 3, "mhd", 1, "fd", HG, "hlle"),
         Case("mhd2d_hg", 2, "mhd", 3, "hg", HG, HG, HG)]


def _set(i, f):
    def change(q):
        q[i] = f(q[i])
    return change


def _vacuum(q):
    q[:] = 0.0
    q[0] = 1.0


# the energy is the variable after the momenta
BREAKS = {"rho_nan": lambda e: _set(0, lambda x: np.nan), "momentum_nan": lambda e: _set(1, lambda x: np.nan),
          "rho_negative": lambda e: _set(0, lambda x: -x), "rho_zero": lambda e: _set(0, lambda x: 0.0),
          "energy_negative": lambda e: _set(e, lambda x: -1.0), "energy_infinite": lambda e: _set(e, lambda x: np.inf),
          "pressure_zero": lambda e: _vacuum}


@pytest.mark.parametrize("np_form", [False, True], ids=["group", "node_parallel"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: c.name)
def test_where_rhs_is_a_number(th, oracle, monkeypatch, case, np_form):
    import torch
    monkeypatch.setenv("TRIXI_HIP_NP_LANES", str(1 << 40) if np_form else "0")
    mesh, cfg = oracle_mesh(oracle, case), oracle_cfg(oracle, case)
    base = oracle.compute_coefficients(cfg, mesh, oracle.IC_SMOOTH_PERIODIC)
    semi = product_semi(th, case)
    try:
        for name, make in BREAKS.items():
            u = base.copy()
            make(case.ndims + 1 if case.equation == "euler" else 4)(u[(3,) + (1,) * case.ndims])
            ref = np.isfinite(oracle.rhs(cfg, mesh, u))
            assert name != "rho_nan" or not ref.all()  # (others stay finite in some fluxes)
            ud = th.pack(torch.from_numpy(u).cuda(), semi)
            du = torch.empty_like(ud)
            th.rhs_hip_(du, ud, semi, 0.0)
            got = np.isfinite(th.wrap_array_native(du, semi).cpu().numpy())
            assert np.array_equal(got, ref), (name, int((~ref).sum()), int((~got).sum()))
    finally:
        semi.close()


@pytest.mark.parametrize("nd,level", [(2, 2), (3, 3)])
def test_max_dt_of_fp32_state(th, nd, level):
    wide = product_semi(th, Case("dt", nd, "euler", level, "fd", "ranocha", ic="smooth_periodic"), "fp64")
    narrow = product_semi(th, Case("dt", nd, "euler", level, "fd", "ranocha", ic="smooth_periodic"), "fp32")
    try:
        u = th.compute_coefficients(0.0, narrow)
        assert th.max_dt(u, narrow) == th.max_dt(u.double(), wide)
    finally:
        wide.close()
        narrow.close()
