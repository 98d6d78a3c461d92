"""The limits of solve()'s native loop, with the library's advance replaced by one
that counts: maxiters of every kind the step-by-step loop takes (steps are taken
while nsteps < maxiters), analysis at its step numbers, step sizes of the user's."""
import math
from types import SimpleNamespace

import pytest
import torch


@pytest.fixture()
def run(th, monkeypatch):
    """run(maxiters, callback) -> (nsteps, chunks): steps of 1/64 towards t = 10^6
    (nobody gets there)."""
    import contextlib
    ti = __import__("sys").modules[th.__name__ + ".time_integration"]
    stream = SimpleNamespace(wait_stream=lambda s: None, synchronize=lambda: None, cuda_stream=1)
    monkeypatch.setattr(torch.cuda, "Stream", lambda: stream)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: stream)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    chunks, single = [], []

    def advance(u, k, t, t_end, semi, cfl=0.0, dt=0.0, max_steps=1, stream=None):
        assert isinstance(max_steps, int) and 1 <= max_steps < 2**63
        assert len(chunks) < 1000, "the loop does not end"
        n = min(max_steps, 32)
        chunks.append(n)
        return t + n * (dt if dt else cfl), n

    def rk_step(u, k, t, dt, semi, use_graph=True, stream=None):
        single.append(dt)

    monkeypatch.setattr(ti, "advance", advance)
    monkeypatch.setattr(ti, "rk_step", rk_step)

    def go(maxiters, callback=(), dt=1 / 64, t1=1e6):
        ode = th.ODEProblem(th.rhs_hip_, torch.zeros(4, dtype=torch.float64), (0.0, t1), SimpleNamespace())
        return th.solve(ode, dt=dt, callback=callback, maxiters=maxiters), chunks, single

    return go


@pytest.mark.parametrize("maxiters,steps", [(0, 0), (1, 1), (7, 7), (100, 100), (2.0, 2), (2.5, 3), (0.5, 1), (-3, 0)])
def test_maxiters(run, maxiters, steps):
    assert run(maxiters)[0].nsteps == steps


@pytest.mark.parametrize("maxiters", [math.inf, 2**63, 2**64, 10**30])
def test_maxiters_without_end(run, maxiters):
    sol = run(maxiters, t1=1.0)[0]
    assert sol.nsteps == 64 and sol.t == 1.0


@pytest.mark.parametrize("interval", [1, 3, 5, 40])
@pytest.mark.parametrize("maxiters", [1, 10, 41, 12.5])
def test_analysis_steps(th, run, monkeypatch, interval, maxiters):
    seen = []
    monkeypatch.setattr(th.AnalysisCallback, "__call__",
                        lambda self, u, t, step, final=False: None if final else seen.append(step))
    run(maxiters, th.AnalysisCallback(None, interval=interval))
    assert [s for s in seen if s % interval == 0] == list(range(interval, math.ceil(maxiters) + 1, interval))


def test_own_step_size(th, run):
    """A step size of the user's, also one set on the instance, is asked every step."""
    cb = th.StepsizeCallback(0.5)
    cb.dt = lambda u, semi: 0.25
    sol, chunks, single = run(6, cb, dt=None)
    assert sol.nsteps == 6 and not chunks and single == [0.25] * 6
