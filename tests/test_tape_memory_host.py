"""The size of the discrete adjoint's tape (CPU only: no kernel is launched, the device's memory
is stubbed)."""
import pytest
import torch

from diffrax_amd import _lib
from diffrax_amd._integrate import ErkPlan


@pytest.fixture(autouse=True)
def gpu_memory(monkeypatch):
    """A stand-in for the device's memory: 100 GiB, all free, no cap on the process."""
    m = dict(free=100 << 30, total=100 << 30, reserved=0, allocated=0, share=1.0)
    stub = lambda name, f: monkeypatch.setattr(torch.cuda, name, f)
    stub("mem_get_info", lambda *a: (m["free"], m["total"]))
    stub("memory_reserved", lambda *a: m["reserved"])
    stub("memory_allocated", lambda *a: m["allocated"])
    stub("get_per_process_memory_fraction", lambda *a: m["share"])
    stub("is_current_stream_capturing", lambda: False)
    return m


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


def test_a_cap_on_the_process_bounds_the_tape(gpu_memory):
    """16 MB of tape: taken from the whole device, from a share of 1 GiB with room, but not
    where it would leave less than 3/4 of that share, whatever the device has free."""
    plan = _plan()
    gpu_memory["share"] = 0.01
    plan.problem.ckpt_every = 64
    assert plan._tape_steps(4096) == 512
    gpu_memory.update(allocated=300 << 20, reserved=300 << 20, free=99 << 30)
    assert plan._tape_steps(4096) == 0
    gpu_memory["share"] = 1.0
    assert plan._tape_steps(4096) == 512


def test_large_tapes_leave_three_quarters_free(gpu_memory):
    plan = _plan(B=65536)
    plan.problem.ckpt_every = 64   # 1 GiB
    assert plan._tape_steps(4096) == 512
    gpu_memory["free"] = 75 << 30
    assert plan._tape_steps(4096) == 0
    gpu_memory["reserved"] = 2 << 30   # cached blocks count as free
    assert plan._tape_steps(4096) == 512


def test_out_of_memory_replays(monkeypatch):
    plan = _plan()
    empty = torch.empty

    def refuse(shape, *a, **k):
        if len(shape) == 4:
            raise torch.OutOfMemoryError("no room")
        return empty(shape, *a, **k)

    monkeypatch.setattr(torch, "empty", refuse)
    plan.record_checkpoints()
    assert plan.problem.ckpt_every == 64 and plan.problem.tape_steps == 0
    assert plan.t["tape"] is None and plan.t["tape_y"] is None and not plan.io.tape
