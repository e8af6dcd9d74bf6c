"""The default solve's own kernel (PID_PLAIN) in workgroups of several waves, whose save times lie
behind one another in LDS, and on every registered field and size, against the general kernel:
the same solve with dtmax = inf, a bound that changes no step, so the same bits."""
import numpy as np
import pytest
import torch

import diffrax_amd as dfx

pytestmark = pytest.mark.gpu


def _solve(cuda, field, args, dtype, solver, y0, t1, ts, launch, dtmax, ckpt):
    plan = dfx._integrate._prepare_erk(
        dfx.ODETerm(field), solver, 0.0, torch.tensor(t1, device=cuda), None,
        torch.tensor(y0, device=cuda, dtype=dtype), args,
        dfx.SaveAt(t0=True, t1=True, ts=torch.tensor(ts, device=cuda)),
        dfx.PIDController(rtol=1e-5, atol=1e-7, dtmax=dtmax), 300, launch)
    if ckpt:
        plan.record_checkpoints()
    plan.launch()
    return [plan.t[k].cpu().numpy().tobytes() for k in ("ys", "ts_out", "stats", "result")]


def _same(cuda, *a, **k):
    for ckpt in (False, True):
        plain, general = (_solve(cuda, *a, dtmax=m, ckpt=ckpt, **k) for m in (None, np.inf))
        assert plain == general, ckpt


# the most save times per instance whose rows fit in a workgroup's 64 KB, and one more
@pytest.mark.parametrize("block,n_ts", [(128, 1), (128, 62), (128, 63), (256, 1), (256, 30),
                                        (256, 31)])
@pytest.mark.parametrize("B", [1, 65, 130, 300])
@pytest.mark.parametrize("shared", [False, True])
def test_workgroups_of_several_waves(cuda, B, block, n_ts, shared):
    rng = np.random.default_rng(B + n_ts)
    t1 = np.full(B, 4.0) if shared else rng.uniform(-6.0, 6.0, B)
    ts = np.sort(rng.uniform(0.0, 1.0, n_ts))
    ts = 4.0 * ts if shared else ts[None] * t1[:, None]
    mu = torch.tensor(rng.uniform(0.1, 5.0, B), device=cuda)
    _same(cuda, dfx.VanDerPol(), mu, torch.float64, dfx.Tsit5(), rng.uniform(-2.0, 2.0, (B, 2)), t1,
          ts, (block, -(-B // block) * block))


@pytest.mark.parametrize("solver", [dfx.Tsit5(), dfx.Dopri5()], ids=repr)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("d", [0, 1, 2, 3, 4, 10])
def test_fields(cuda, d, dtype, solver):
    """Lotka-Volterra (d = 0 here) and the linear fields, whose error norms differ with d."""
    B, n_ts = 70, 9
    rng = np.random.default_rng(d)
    t1 = rng.uniform(0.0, 3.0, B)
    t1[3] = 0.0
    ts = np.linspace(0.0, 1.0, n_ts)[None] * t1[:, None]
    ts[:, -1] = t1
    if d == 0:
        field, args, y0 = dfx.LotkaVolterra(), (1.5, 1.0, 3.0, 1.0), rng.uniform(0.5, 2.0, (B, 2))
    else:
        A = rng.normal(size=(d, d)) - 2.0 * np.eye(d)
        field, args = dfx.LinearField(), torch.tensor(A, device=cuda, dtype=dtype)
        y0 = rng.normal(size=(B, d))
        y0[5, 0] = np.nan
        y0[7] = 0.0
    _same(cuda, field, args, dtype, solver, y0, t1, ts, None)
