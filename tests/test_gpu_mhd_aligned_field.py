"""GLM-MHD where the field lies along a coordinate direction and the Alfven speed
equals the sound speed (gamma p = |B|^2): the fast speed's inner root is zero there,
and formed as a difference it rounds below zero and gives NaN.  A uniform state is a
steady state, and its speeds are known: c_f^2 = gamma p / rho along the field, twice
that across it."""
import numpy as np
import pytest

from cases import Case, product_semi

pytestmark = pytest.mark.gpu

EPS = {"fp64": 2.0**-52, "mixed": 2.0**-23}


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _states(gamma):
    """Uniform states (rho, rho v, rho e, B, psi) with gamma p = |B|^2, B along x, y or z."""
    rng = np.random.default_rng(20261205)
    for i in range(24):
        rho, b = rng.uniform(0.3, 3.0), rng.uniform(0.2, 2.0) * rng.choice([-1.0, 1.0])
        v, B = rng.uniform(-0.5, 0.5, 3), np.zeros(3)
        B[i % 3] = b
        p = b * b / gamma
        e = p / (gamma - 1) + 0.5 * rho * v @ v + 0.5 * b * b
        yield rho, v, p, i % 3, np.array([rho, *(rho * v), e, *B, 0.0])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("ndims,vi,sflux", [(2, "fd", "llf"), (3, "fd", "llf"), (2, "fd", "llf_naive"), (3, "fd", "hlle"),
                                            (2, "fd", "hlle"), (2, "hg", "llf")])
def test_uniform_state(th, torch, ndims, vi, sflux, precision):
    gamma, length = 5.0 / 3.0, 4.0
    case = Case("aligned", ndims, "mhd", 1 if ndims == 3 else 2, vi, "hindenlang_gassner", sflux, "llf", gamma=gamma,
                ic="smooth_periodic", precision=precision)
    semi = product_semi(th, case)
    scale = 2.0 / (length / 2**case.level)  # inverse Jacobian
    try:
        for rho, v, p, axis, q in _states(gamma):
            u = th.pack(torch.from_numpy(np.broadcast_to(q, semi.trixi_shape).copy()).cuda(), semi)
            du = torch.empty_like(u)
            th.rhs_hip_(du, u, semi, 0.0)
            got = float(du.abs().max())
            # some 30 terms of fluxes below 2 (|q| + c |q|) with weights below 6 of which each
            # is rounded a few times
            speed = abs(v).max() + np.sqrt(2.0 * gamma * p / rho)
            bound = 30 * 6 * 8 * EPS[precision] * scale * 2.0 * (1.0 + speed) * np.abs(q).max()
            assert got <= bound, (axis, q, got, bound)
            # max_dt is computed in FP64
            lam = sum(abs(v[d]) + np.sqrt((1.0 if d == axis else 2.0) * gamma * p / rho) for d in range(ndims))
            dt = th.max_dt(u, semi)
            # at the root's zero an error e in its argument is one of sqrt(e) in it: sqrt(a few 2^-52)
            assert abs(dt * (4 * scale * lam) / 2.0 - 1.0) < 1e-7, (axis, q, dt)
    finally:
        semi.close()
