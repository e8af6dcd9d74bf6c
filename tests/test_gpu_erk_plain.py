"""The default solve's own kernel (ErkLane with PID_PLAIN: save times in LDS, controller
options resolved at compile time) against the general one, which the same solve takes with
dtmax = inf: that bound changes no step, so rows, times, counters and results are the same
bits, also for solves that blow up, start at NaN or inf, take no step or run backwards."""
import numpy as np
import pytest
import torch

import diffrax_amd as dfx

pytestmark = pytest.mark.gpu


def _solve(cuda, dtype, solver, y0, mu, t1, ts, n_steps, dtmax, ckpt):
    ctrl = dfx.PIDController(rtol=1e-5, atol=1e-7, dtmax=dtmax)
    saveat = dfx.SaveAt(t0=True, t1=True) if ts is None else dfx.SaveAt(
        ts=torch.tensor(ts, device=cuda), t1=True)
    plan = dfx._integrate._prepare_erk(
        dfx.ODETerm(dfx.VanDerPol()), solver, 0.0, torch.tensor(t1, device=cuda), None,
        torch.tensor(y0, device=cuda, dtype=dtype), torch.tensor(mu, device=cuda, dtype=dtype),
        saveat, ctrl, n_steps, None)
    if ckpt:
        plan.record_checkpoints()
    plan.launch()
    return [plan.t[k].cpu().numpy().tobytes() for k in ("ys", "ts_out", "stats", "result")]


# n_ts: none, one, a few, the most whose rows fit in a workgroup's LDS (126) and one more
@pytest.mark.parametrize("n_ts", [0, 1, 7, 126, 127])
@pytest.mark.parametrize("B", [1, 63, 65, 130])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_same_bits_as_general(cuda, dtype, B, n_ts):
    rng = np.random.default_rng(B * 1000 + n_ts)
    y0 = rng.uniform(-2.0, 2.0, (B, 2))
    mu = rng.uniform(0.1, 5.0, B)
    t1 = rng.uniform(-6.0, 6.0, B)
    if B > 60:
        t1[5] = 0.0                                    # no step
        y0[7] = [1e30, -1e30]                          # blows up
        y0[9, 1] = np.nan
        y0[11, 0] = np.inf
        mu[13] = 1e6                                   # rejected steps until max_steps
    ts = np.linspace(0.0, 1.0, n_ts)[None] * t1[:, None] if n_ts else None
    if n_ts:
        ts[:, -1] = t1
    for solver in (dfx.Tsit5(), dfx.Dopri5()):
        for ckpt in (False, True):
            a = _solve(cuda, dtype, solver, y0, mu, t1, ts, 300, None, ckpt)
            b = _solve(cuda, dtype, solver, y0, mu, t1, ts, 300, np.inf, ckpt)
            assert a == b, (solver, ckpt)


@pytest.mark.parametrize("n_ts", [1, 65, 1000])
@pytest.mark.parametrize("B", [1, 65])
def test_shared_times_same_bits_as_general(cuda, B, n_ts):
    rng = np.random.default_rng(n_ts)
    y0 = rng.uniform(-2.0, 2.0, (B, 2))
    mu = rng.uniform(0.1, 2.0, B)
    ts = np.sort(rng.uniform(0.0, 4.0, n_ts))
    t1 = np.full(B, 4.0)
    a, b = (_solve(cuda, torch.float64, dfx.Dopri5(), y0, mu, t1, ts, 4096, m, False)
            for m in (None, np.inf))
    assert a == b


def test_more_waves_than_simds(cuda):
    """One instance past 65,536: the build without a SIMD per wave."""
    B = 65537
    rng = np.random.default_rng(7)
    y0 = rng.uniform(-2.0, 2.0, (B, 2))
    mu = rng.uniform(0.1, 2.0, B)
    t1 = rng.uniform(0.5, 2.0, B)
    ts = np.stack([np.zeros(B), 0.5 * t1, t1], axis=1)
    for ckpt in (False, True):
        a, b = (_solve(cuda, torch.float64, dfx.Tsit5(), y0, mu, t1, ts, 256, m, ckpt)
                for m in (None, np.inf))
        assert a == b, ckpt
