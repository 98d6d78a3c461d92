"""States in other units: density scaled by A, pressure by B, velocities by
sqrt(B / A) (and the field by sqrt(B)), all powers of two, so that every quantity
of the rhs! scales exactly and only its exponent changes.  The result must be that
of the unscaled state as long as the quantities themselves (rho, p, rho p, squares
of speeds) lie inside the FP64 range, also where rho^2 p does not."""
import numpy as np
import pytest

from cases import Case, product_semi, rel_max

pytestmark = pytest.mark.gpu

# log2 of (A, B): rho^2 p = 2^-1100 (zero in FP64), 2^1100 (infinite), and ordinary units
SCALES = [(-400, -300), (400, 300), (-450, -150), (-60, 40)]
HG = "hindenlang_gassner"


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _scales(case, a, b):
    """log2 factors of (state, du) per variable."""
    v = (b - a) // 2
    if case.equation == "euler":
        u = [a] + [a + v] * case.ndims + [b]
    else:
        u = [a] + [a + v] * 3 + [b] + [b // 2] * 4
    return np.array(u), np.array(u) + v


def _pow2(torch, e):
    return torch.tensor([2.0**int(x) for x in e], dtype=torch.float64, device="cuda")


CASES = [(2, "euler", 3, "fd", "ranocha", "llf", "smooth_periodic"), (3, "euler", 2, "fd", "ranocha", "llf", "smooth_periodic"),
         (3, "euler", 2, "fd", "ranocha", "ranocha", "smooth_periodic"), (2, "euler", 3, "fd", "ranocha", "ranocha", "seeded_random"),
         (3, "euler", 2, "fd", "shima_etal", "llf", "smooth_periodic"), (2, "euler", 4, "hg", "ranocha", "llf", "weak_blast_wave"),
         (3, "mhd", 2, "fd", HG, "llf", "smooth_periodic"), (2, "mhd", 3, "fd", HG, HG, "smooth_periodic")]


@pytest.mark.parametrize("np_lanes", ["0", ""], ids=["lane_groups", "by_size"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_rhs_of_scaled_state(th, torch, monkeypatch, case, np_lanes):
    nd, eq, level, vi, vflux, sflux, ic = case
    if np_lanes:
        monkeypatch.setenv("TRIXI_HIP_NP_LANES", np_lanes)
    ref = None
    for a, b in [(0, 0)] + SCALES:
        # (the cleaning speed is a speed)
        c = Case("scaled", nd, eq, level, vi, vflux, sflux, "llf", ic=ic, c_h=2.0**((b - a) // 2), indicator="density")
        semi = product_semi(th, c)
        try:
            if ref is None:
                base = th.compute_coefficients(0.0, semi)
            su, sdu = (_pow2(torch, e).reshape(-1, 1, 1) for e in _scales(c, a, b))
            u = (base.view(semi.native_shape) * su).reshape(-1)
            du = torch.empty_like(u)
            th.rhs_hip_(du, u, semi, 0.0)
            got = (du.view(semi.native_shape) / sdu).cpu().numpy()
        finally:
            semi.close()
        if ref is None:
            ref = got
            assert np.isfinite(ref).all()
        # another path through the logarithmic means may round differently: the parity bound
        err = rel_max(got, ref)
        assert err <= 1e-12, (a, b, err)


@pytest.mark.parametrize("nd,level,sflux", [(3, 2, "llf"), (2, 3, "ranocha"), (3, 3, "ranocha")])
def test_vjp_of_scaled_state(th, torch, monkeypatch, nd, level, sflux):
    """The adjoint takes 1 / (rho p)^2 too, so rho^2 p leaves the range first only
    where p is large and rho small, or the reverse."""
    monkeypatch.setenv("TRIXI_HIP_VJP_PD_LANES", "0")  # lane groups on every mesh
    ref = None
    for a, b in ((0, 0), (-650, 200), (650, -200), (600, -100), (-60, 40)):
        semi = product_semi(th, Case("scaled", nd, "euler", level, "fd", "ranocha", sflux, ic="smooth_periodic"))
        try:
            th.enable_adjoint(semi)
            eu, edu = _scales(Case("scaled", nd, "euler", level), a, b)
            su, sv = _pow2(torch, eu).reshape(-1, 1, 1), _pow2(torch, -edu).reshape(-1, 1, 1)
            u = (th.compute_coefficients(0.0, semi).view(semi.native_shape) * su).reshape(-1)
            i = torch.arange(u.numel(), device="cuda", dtype=torch.float64)
            vbar = (torch.cos(i).view(semi.native_shape) * sv).reshape(-1)
            out = torch.zeros_like(u)
            got = (th.rhs_vjp(out, u, vbar, semi).view(semi.native_shape) * su).cpu().numpy()
        finally:
            semi.close()
        if ref is None:
            ref = got
            assert np.isfinite(ref).all()
        err = rel_max(got, ref)
        assert err <= 1e-12, (a, b, err)
