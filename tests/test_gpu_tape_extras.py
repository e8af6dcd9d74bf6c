"""The discrete adjoint of forward solves that also export their state (state_out) or dense
output.  Their kernels write no tape (dfx_erk_io.tape): a problem that declares one is refused,
and without one the adjoint replays, to the same gradient bits."""
import ctypes

import numpy as np
import pytest
import torch

import diffrax_amd as dfx
from diffrax_amd import _lib

pytestmark = pytest.mark.gpu


def _plan(cuda, B, ctrl, **saves):
    rng = np.random.default_rng(B)
    y0 = torch.tensor(rng.uniform(-2.0, 2.0, (B, 2)), device=cuda)
    mu = torch.tensor(rng.uniform(0.2, 4.0, B), device=cuda)
    plan = dfx._integrate._prepare_erk(
        dfx.ODETerm(dfx.VanDerPol()), dfx.Tsit5(), 0.0, 3.0, 0.05, y0, mu,
        dfx.SaveAt(ts=torch.linspace(0.0, 3.0, 6, dtype=torch.float64), **saves), ctrl, 256, None)
    plan.record_checkpoints()
    return plan


@pytest.mark.parametrize("ctrl", [dfx.PIDController(rtol=1e-5, atol=1e-7),
                                  dfx.PIDController(rtol=1e-5, atol=1e-7, pcoeff=0.2, icoeff=0.8),
                                  dfx.ConstantStepSize()],
                         ids=["default", "pi", "constant"])
@pytest.mark.parametrize("B", [1, 65])
def test_gradient_of_solves_with_extras(cuda, B, ctrl):
    grads = []
    for saves in ({}, dict(solver_state=True), dict(dense=True)):
        plan = _plan(cuda, B, ctrl, **saves)
        assert plan.problem.tape_steps == (0 if saves else 128)
        plan.launch()
        yb = torch.empty((B, 2), dtype=torch.float64, device=cuda)
        qb = torch.empty((B, 1), dtype=torch.float64, device=cuda)
        plan.adjoint((2.0 * plan.t["ys"]).contiguous(), yb, qb)
        assert int(plan.t["stats"][:, 0].max()) <= 128   # on the tape where there is one
        grads.append((yb, qb))
    assert bool((grads[0][1] != 0).all())
    for yb, qb in grads[1:]:
        assert torch.equal(yb, grads[0][0]) and torch.equal(qb, grads[0][1])


@pytest.mark.parametrize("saves", [dict(solver_state=True), dict(dense=True)], ids=["state", "dense"])
def test_a_tape_that_stays_unwritten_is_refused(cuda, saves):
    """Through the C ABI, as a caller who declares a tape for every solve."""
    plan = _plan(cuda, 65, dfx.PIDController(rtol=1e-5, atol=1e-7), **saves)
    tape = torch.zeros((2, 128, 64, 4), dtype=torch.float64, device=cuda)
    plan.problem.tape_steps = 128
    plan.io.tape, plan.io.tape_y = tape[..., :2].data_ptr(), tape[..., 2:].data_ptr()
    rc = _lib.load().dfx_erk_solve(
        ctypes.byref(plan.problem), ctypes.byref(plan.io), ctypes.c_void_p(plan.ws.data_ptr()),
        ctypes.c_size_t(plan.ws.numel()), None, torch.cuda.current_stream().cuda_stream)
    assert rc != 0
    plan.problem.tape_steps = 0
    plan.launch()
    assert bool(torch.isfinite(plan.t["ys"]).all())
