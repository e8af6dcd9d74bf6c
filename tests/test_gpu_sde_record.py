"""The SDE gradient with saves at t0 and t1 by its two records, forward sensitivities and
checkpoints (which a small given number of checkpoints selects): the same gradient."""
import numpy as np
import pytest
import torch

import diffrax_amd as dfx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("N", [3, 100])
def test_records_agree(cuda, dtype, N):
    rng = np.random.default_rng(N)
    P, d = 70, 8
    cast = lambda a: torch.tensor(a, device=cuda, dtype=dtype)
    dW = torch.tensor(rng.normal(size=(N, P, d)) / np.sqrt(N), device=cuda, dtype=torch.float32)
    y0, w = cast(rng.normal(size=(P, d))), cast(rng.normal(size=(P, 2, d)))
    par = [cast(a) for a in (rng.uniform(0.5, 2.0, d), rng.normal(size=d),
                             rng.uniform(0.1, 0.5, d))]
    terms = dfx.MultiTerm(dfx.ODETerm(dfx.OUDrift()),
                          dfx.ControlTerm(dfx.DiagonalNoise(), dfx.IncrementPath(dW)))
    grads = []
    for checkpoints in (None, 1):
        leaves = [a.clone().requires_grad_() for a in (y0, *par)]
        sol = dfx.diffeqsolve(terms, dfx.Heun(), 0.0, 1.0, 1.0 / N, leaves[0], tuple(leaves[1:]),
                              saveat=dfx.SaveAt(t0=True, t1=True),
                              stepsize_controller=dfx.ConstantStepSize(),
                              adjoint=dfx.RecursiveCheckpointAdjoint(checkpoints=checkpoints))
        grads.append(torch.autograd.grad((sol.ys * w).sum(), leaves))
    tol = (N + 4) * torch.finfo(dtype).eps   # a rounding per step and four per term
    for a, b in zip(*grads):
        scale = w.abs().sum(0).max() if a.ndim == 1 else 1.0
        assert float((a - b).abs().max()) <= tol * max(float(scale), float(a.abs().max()))
