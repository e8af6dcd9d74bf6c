"""SaveAt(ts) rows of the neural-ODE kernel, whose owner threads take a group of save times at
once (8 or 16, by the wave count): counts per step around the group size, repeated times,
times on step ends, per-trajectory rows.  Each row equals the dense output evaluated at its
time, bit for bit (the dense evaluation's arithmetic is the solve's)."""
import numpy as np
import pytest
import torch

import diffrax_amd as dfx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("matmul", ["f32", "bf16"])
@pytest.mark.parametrize("launch", [4, 8])
@pytest.mark.parametrize("n_ts", [1, 7, 8, 9, 15, 16, 17, 64, 200])
def test_rows_equal_the_dense_output(cuda, matmul, launch, n_ts):
    rng = np.random.default_rng(n_ts)
    shapes = [(256, 64), (256,), (256, 256), (256,), (64, 256), (64,)]
    P = [rng.normal(0.0, np.sqrt(2.0 / sum(s)) if len(s) == 2 else 0.1, size=s) for s in shapes]
    term = dfx.ODETerm(dfx.MLPField(
        *[torch.tensor(p, dtype=torch.float32, device=cuda) for p in P], matmul=matmul))
    B = 35
    y0 = torch.tensor(rng.normal(size=(B, 64)), dtype=torch.float32, device=cuda)
    kw = dict(stepsize_controller=dfx.PIDController(rtol=1e-5, atol=1e-7), max_steps=64,
              launch=launch)
    dense = dfx.diffeqsolve(term, dfx.Tsit5(), 0.0, 1.0, 0.1, y0,
                            saveat=dfx.SaveAt(t1=True, dense=True), **kw)
    ts = np.sort(rng.uniform(0.0, 1.0, size=(B, n_ts)), axis=1)
    ts[:, n_ts // 2:n_ts // 2 + 3] = ts[:, n_ts // 2:n_ts // 2 + 1]      # repeated
    knots = dense.interpolation.plan.dense["dense_ts"][:, 1].cpu().numpy()
    ts[:, 0] = np.minimum(ts[:, 0], knots)
    ts = np.sort(np.where(np.arange(n_ts) == n_ts // 3, knots[:, None], ts), axis=1)
    ts = torch.tensor(ts, dtype=torch.float64, device=cuda)
    sol = dfx.diffeqsolve(term, dfx.Tsit5(), 0.0, 1.0, 0.1, y0,
                          saveat=dfx.SaveAt(t0=True, t1=True, ts=ts), **kw)
    assert torch.equal(sol.stats["num_steps"], dense.stats["num_steps"])
    assert torch.equal(sol.ts[:, 1:-1], ts)
    assert torch.equal(sol.ys[:, 1:-1], dense.evaluate(ts))
    assert torch.equal(sol.ys[:, 0], y0) and torch.equal(sol.ys[:, -1], dense.ys[:, -1])
