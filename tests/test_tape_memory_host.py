"""The size of the discrete adjoint's tape (CPU only: no kernel is launched)."""

import pytest
import torch

from diffrax_amd import _lib
from diffrax_amd._integrate import ErkPlan


def _plan(B=1000, d=2, dtype=torch.float64, max_steps=4096):
    plan = ErkPlan.__new__(ErkPlan)
    plan.problem = _lib.ErkProblem(d=d, max_steps=max_steps, batch=B)
    plan.t = {"y0": torch.zeros((B, d), dtype=dtype)}
    plan.io = _lib.ErkIO()
    return plan


def _bytes(t):
    return 0 if t is None else t.numel() * t.element_size()


@pytest.mark.parametrize("checkpoints", [1, 2, 5, 16, 64, 200, 4096])
@pytest.mark.parametrize("d,dtype", [(2, torch.float64), (2, torch.float32), (4, torch.float64)])
def test_a_given_number_of_checkpoints_bounds_the_tape(checkpoints, d, dtype):
    plan = _plan(B=128, d=d, dtype=dtype)
    plan.record_checkpoints(checkpoints)
    tape = _bytes(plan.t["tape"]) + _bytes(plan.t["tape_y"])
    assert tape <= _bytes(plan.t["ckpt"])
    assert (plan.problem.tape_steps > 0) == (tape > 0)
    if checkpoints >= 64:
        assert plan.problem.tape_steps >= 2 * plan.problem.ckpt_every


def test_default_tape():
    plan = _plan()
    plan.record_checkpoints()
    assert plan.problem.ckpt_every == 64 and plan.problem.tape_steps == 512
