"""The SDE gradient with saves at t0 and t1 only (sde_heun_sens_kernel)."""
import math

import numpy as np
import pytest
import torch

import diffrax_amd as dfx
from diffrax_amd import _sde

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("P,d,N", [(1, 4, 1), (3, 4, 15), (65, 8, 16), (17, 256, 17),
                                   (1025, 16, 33), (40, 32, 257), (9000, 16, 3)])
def test_sde_t1_gradient_without_a_second_pass(cuda, dtype, P, d, N):
    """Saves at t0 and t1 only: the forward carries dy(t1)/dtheta and dy(t1)/dsigma, and the
    backward reduces them.  Against torch float64 autograd through the same Heun steps, at
    the edges of the load groups (16 steps), the workgroups (256 threads) and the backward's
    grid (512 blocks).  Normwise bound: one rounding per step and 4 in forming each term, in
    the state's precision."""
    rng = np.random.default_rng(P + N)
    th, mu, sg = rng.uniform(0.5, 2.0, d), rng.normal(size=d), rng.uniform(0.1, 0.5, d)
    cast = lambda a: torch.tensor(a).to(dtype)
    dW = torch.tensor(rng.normal(size=(N, P, d)) * math.sqrt(1.0 / N), dtype=torch.float32)
    y0, wt = cast(rng.normal(size=(P, d))), cast(rng.normal(size=(P, 2, d)))
    leaves = [cast(a).to(cuda).requires_grad_() for a in (th, mu, sg)]
    y0g = y0.to(cuda).requires_grad_()
    sol = dfx.diffeqsolve(
        dfx.MultiTerm(dfx.ODETerm(dfx.OUDrift()),
                      dfx.ControlTerm(dfx.DiagonalNoise(), dfx.IncrementPath(dW.to(cuda)))),
        dfx.Heun(), 0.0, 1.0, 1.0 / N, y0g, tuple(leaves),
        saveat=dfx.SaveAt(t0=True, t1=True), stepsize_controller=dfx.ConstantStepSize())
    got = torch.autograd.grad((sol.ys * wt.to(cuda)).sum(), [y0g, *leaves])

    ref = [cast(a).double().requires_grad_() for a in (th, mu, sg)]
    y0r = y0.double().requires_grad_()
    grid = _sde.constant_grid(0.0, 1.0, 1.0 / N)
    y = y0r
    for n in range(N):
        dt, w = float(grid[n + 1] - grid[n]), ref[2] * dW[n].double()
        k0 = dt * (ref[0] * (ref[1] - y)) + w
        k1 = dt * (ref[0] * (ref[1] - (y + k0))) + w
        y = y + 0.5 * (k0 + k1)
    want = torch.autograd.grad((torch.stack([y0r, y], 1) * wt.double()).sum(), [y0r, *ref])
    tol = (N + 4) * torch.finfo(dtype).eps
    for g, r in zip(got, want):
        scale = r.abs().max().clamp_min(wt.double().abs().sum(0).max() if r.ndim == 1 else 1.0)
        assert (g.double().cpu() - r).abs().max() <= tol * scale
