"""The tape of attempted steps that the discrete adjoint sweeps (dfx_erk_io.tape): a solve
whose steps fit on it, one that outgrows it and one without it take the same steps with the
same arithmetic, so their gradients are the same bits, those of the oracle's adjoint."""
import numpy as np
import pytest
import torch

import diffrax_amd as dfx
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 64, 130])
@pytest.mark.parametrize("solver", [dfx.Tsit5(), dfx.Dopri5(), dfx.Heun()], ids=repr)
def test_tape_and_replay_same_bits(cuda, solver, B):
    rng = np.random.default_rng(5 + B)
    y0 = rng.uniform(-2.0, 2.0, (B, 2))
    mu = rng.uniform(0.2, 4.0, (B, 1))
    t1 = rng.uniform(0.5, 6.0, B)
    t1[B // 2] = 0.0 if B > 1 else t1[0]          # a solve of no steps among the others
    ts = np.linspace(0.0, 1.0, 5)[None] * t1[:, None]
    ts[:, -1] = t1
    grads, counts = [], None
    for tape in (None, 0, "short"):
        plan = dfx._integrate._prepare_erk(
            dfx.ODETerm(dfx.VanDerPol()), solver, 0.0, torch.tensor(t1, device=cuda), 0.05,
            torch.tensor(y0, device=cuda), torch.tensor(mu, device=cuda)[:, 0],
            dfx.SaveAt(t0=True, ts=torch.tensor(ts, device=cuda), t1=True),
            dfx.PIDController(rtol=1e-5, atol=1e-7), 4096, None)
        plan.record_checkpoints()
        assert plan.problem.ckpt_every == 64 and plan.problem.tape_steps == 512
        if tape is not None:
            # the length of the longest solve less one: its workgroup replays, others do not
            n = 0 if tape == 0 else int(counts.max()) - 1
            plan.problem.tape_steps = n
            plan.t["tape"] = torch.empty((-(-B // 64), max(n, 1), 64, 2), dtype=torch.float64, device=cuda)
            plan.t["tape_y"] = torch.empty((-(-B // 64), max(n, 1), 64, 2), dtype=torch.float64, device=cuda)
            plan._bind()
        plan.launch()
        yb = torch.empty((B, 2), dtype=torch.float64, device=cuda)
        qb = torch.empty((B, 1), dtype=torch.float64, device=cuda)
        plan.adjoint((2.0 * plan.t["ys"]).contiguous(), yb, qb)
        counts = plan.t["stats"][:, 0].cpu().numpy()
        grads.append((yb.cpu().numpy(), qb.cpu().numpy()))
    # Heun outgrows the default tape too, the fifth-order solvers fit on it
    assert counts.max() > 1 and (isinstance(solver, dfx.Heun) or counts.max() <= 512)
    for yb, qb in grads[1:]:
        assert np.array_equal(yb, grads[0][0]) and np.array_equal(qb, grads[0][1])
    kw = dict(solver=type(solver).__name__.lower(), vf="vdp", dt0=0.05, rtol=1e-5, atol=1e-7,
              max_steps=4096)
    fwd = oracle.solve(y0, t1, mu, ts=ts, save_t0=True, save_t1=True, record_grid=True, **kw)
    ryb, rqb = oracle.adjoint(t1, mu, fwd, 2.0 * fwd["ys"], ts=ts, save_t0=True, save_t1=True, **kw)
    assert np.array_equal(grads[0][0], ryb) and np.array_equal(grads[0][1], rqb)


@pytest.mark.parametrize("B", [65536, 65537])
def test_tape_one_and_two_waves_per_simd(cuda, B):
    """The sweep's builds with and without a SIMD per wave, against the replay."""
    gen = torch.Generator(device=cuda).manual_seed(3)
    y0 = torch.rand(B, 2, generator=gen, device=cuda, dtype=torch.float64) * 2 - 1
    mu = torch.rand(B, generator=gen, device=cuda, dtype=torch.float64) + 0.2
    t1 = torch.rand(B, generator=gen, device=cuda, dtype=torch.float64) + 0.5
    out = []
    for tape in (True, False):
        plan = dfx._integrate._prepare_erk(
            dfx.ODETerm(dfx.VanDerPol()), dfx.Tsit5(), 0.0, t1, 0.1, y0, mu,
            dfx.SaveAt(ts=torch.stack([0.5 * t1, t1], 1)), dfx.PIDController(rtol=1e-5, atol=1e-7),
            256, None)
        plan.record_checkpoints()
        assert plan.problem.tape_steps == 128
        if not tape:
            plan.problem.tape_steps = 0
        plan.launch()
        yb = torch.empty((B, 2), dtype=torch.float64, device=cuda)
        qb = torch.empty((B, 1), dtype=torch.float64, device=cuda)
        plan.adjoint((2.0 * plan.t["ys"]).contiguous(), yb, qb)
        out.append((yb, qb))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    assert bool(torch.isfinite(out[0][0]).all())
