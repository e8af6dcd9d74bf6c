"""The discrete adjoint's tape (dfx_erk_io.tape) of forward solves that also export their state
(state_out) or dense output: the same steps as without, so the same gradient bits, whether the
adjoint sweeps the tape or replays."""
import numpy as np
import pytest
import torch

import diffrax_amd as dfx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ctrl", [dfx.PIDController(rtol=1e-5, atol=1e-7),
                                  dfx.PIDController(rtol=1e-5, atol=1e-7, pcoeff=0.2, icoeff=0.8),
                                  dfx.ConstantStepSize()],
                         ids=["default", "pi", "constant"])
@pytest.mark.parametrize("B", [1, 65])
def test_gradient_of_solves_with_extras(cuda, B, ctrl):
    rng = np.random.default_rng(B)
    y0 = torch.tensor(rng.uniform(-2.0, 2.0, (B, 2)), device=cuda)
    mu = torch.tensor(rng.uniform(0.2, 4.0, B), device=cuda)
    ts = torch.linspace(0.0, 3.0, 6, dtype=torch.float64)
    grads = []
    for saves, tape in (({}, False), ({}, True), (dict(solver_state=True), True),
                        (dict(solver_state=True), False), (dict(dense=True), True)):
        plan = dfx._integrate._prepare_erk(
            dfx.ODETerm(dfx.VanDerPol()), dfx.Tsit5(), 0.0, 3.0, 0.05, y0, mu,
            dfx.SaveAt(ts=ts, **saves), ctrl, 256, None)
        plan.record_checkpoints()
        assert plan.problem.tape_steps == 128
        if tape:
            plan.t["tape"].zero_()   # a forward that leaves it unwritten shows
            plan.t["tape_y"].zero_()
        else:
            plan.problem.tape_steps = 0
        plan.launch()
        yb = torch.empty((B, 2), dtype=torch.float64, device=cuda)
        qb = torch.empty((B, 1), dtype=torch.float64, device=cuda)
        plan.adjoint((2.0 * plan.t["ys"]).contiguous(), yb, qb)
        assert int(plan.t["stats"][:, 0].max()) <= 128   # on the tape
        grads.append((yb, qb))
    assert bool((grads[0][1] != 0).all())
    for yb, qb in grads[1:]:
        assert torch.equal(yb, grads[0][0]) and torch.equal(qb, grads[0][1])
