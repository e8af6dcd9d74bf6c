"""Times that require a gradient are refused, on the host and on a device (CPU only: meta tensors
stand for the device's; the refusal comes before any GPU work)."""
import pytest
import torch

import diffrax_amd as dfx
from diffrax_amd import _mlp
from diffrax_amd._integrate import _prepare_erk

CTRL = dfx.PIDController(rtol=1e-5, atol=1e-7)


def _times(device, grad=True, n=3):
    return torch.linspace(0.0, 1.0, n, dtype=torch.float64, device=device).requires_grad_(grad)


def _erk(t1, ts):
    return _prepare_erk(dfx.ODETerm(dfx.VanDerPol()), dfx.Tsit5(), 0.0, t1, 0.1,
                        torch.zeros((3, 2), dtype=torch.float64), 1.0, dfx.SaveAt(ts=ts), CTRL,
                        100, None)


@pytest.mark.parametrize("t1,ts", [(1.0, "cpu"), (1.0, "meta"), ("cpu", "meta-"), ("meta", "cpu-"),
                                   ("meta-", "cpu"), ("meta-", "meta"), ("meta", "meta-")])
def test_small_systems(t1, ts):
    make = lambda s: _times(s.rstrip("-"), not s.endswith("-")) if isinstance(s, str) else s
    with pytest.raises(RuntimeError, match="gradients with respect to t1"):
        _erk(make(t1), make(ts))


@pytest.mark.parametrize("ts", ["cpu", "meta"])
def test_neural_ode(ts):
    shapes = ((256, 64), (256,), (256, 256), (256,), (64, 256), (64,))
    field = dfx.MLPField(*(torch.zeros(s) for s in shapes))
    with pytest.raises(RuntimeError, match="gradients with respect to t1"):
        _mlp.prepare_mlp(dfx.ODETerm(field), dfx.Tsit5(), 0.0, 1.0, 0.1, torch.zeros((3, 64)),
                         dfx.SaveAt(ts=_times(ts)), CTRL, 100, torch.device("cpu"))


def test_without_gradients_host_times_stay_refused():
    with torch.no_grad(), pytest.raises(RuntimeError):
        _erk(_times("meta", False), _times("cpu"))
