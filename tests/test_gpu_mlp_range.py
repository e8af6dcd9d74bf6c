"""Gradients of the neural ODE where layer inputs, deltas or weights are outside the range that
three bfloat16 pieces hold (SplitRange): infinities of a piece, and magnitudes whose low pieces
vanish.  The float32 form and the weight-gradient GEMM take float32 MFMA there, so a gradient is
as good as inside the range.  Bound of each comparison, normwise: both sides are within 1e-6 of
the float64 gradient (float32 sums of a few hundred terms), so they are within 3e-6 of each
other."""
import numpy as np
import pytest
import torch

import diffrax_amd as dfx
from tests.test_gpu_mlp_grad import _weights

pytestmark = pytest.mark.gpu

TOL = 3e-6
BACK = dfx.BacksolveAdjoint(stepsize_controller=dfx.PIDController(
    rtol=1e-5, atol=1e-7, norm=dfx.adjoint_rms_seminorm))


# equal backward steps whatever the cotangents' size
EVEN = dfx.BacksolveAdjoint(dt0=-0.125, stepsize_controller=dfx.PIDController(
    rtol=1.0, atol=1.0, dtmax=0.125, norm=dfx.adjoint_rms_seminorm))


def _grads(cuda, matmul, W, y0, w, adjoint=dfx.RecursiveCheckpointAdjoint()):
    P = [torch.tensor(a, dtype=torch.float32, device=cuda, requires_grad=True) for a in W]
    y0 = torch.tensor(y0, device=cuda, requires_grad=True)
    sol = dfx.diffeqsolve(dfx.ODETerm(dfx.MLPField(*P, matmul=matmul)), dfx.Tsit5(), 0.0, 1.0,
                          0.1, y0, saveat=dfx.SaveAt(ts=np.linspace(0.0, 1.0, w.shape[1])),
                          stepsize_controller=dfx.PIDController(rtol=1e-5, atol=1e-7),
                          adjoint=adjoint)
    g = torch.autograd.grad(sol.ys, [y0, *P], torch.tensor(w, device=cuda))
    return [a.double().cpu() for a in g]


def _close(got, want):
    for name, g, r in zip(("y0", "W1", "b1", "W2", "b2", "W3", "b3"), got, want):
        err = float((g - r).abs().max() / r.abs().max())
        assert err < TOL, (name, err)


def _inputs(B=70):
    rng = np.random.default_rng(3)
    y0 = rng.normal(size=(B, 64)).astype(np.float32)
    return y0, rng.normal(size=(B, 5, 64)).astype(np.float32)


@pytest.mark.parametrize("adjoint", [dfx.RecursiveCheckpointAdjoint(), EVEN],
                         ids=["discrete", "backsolve"])
@pytest.mark.parametrize("e", [-104, -112, -116])
def test_small_cotangents(cuda, e, adjoint):
    """The gradient is linear in the cotangents, also where these are near the least number."""
    W, (y0, w) = _weights(), _inputs()
    s = np.float32(2.0 ** e)
    got = _grads(cuda, "f32", W, y0, w * s, adjoint)
    _close([g / float(s) for g in got], _grads(cuda, "f32", W, y0, w, adjoint))


@pytest.mark.parametrize("adjoint", [dfx.RecursiveCheckpointAdjoint(), BACK],
                         ids=["discrete", "backsolve"])
def test_large_state(cuda, adjoint):
    """A state near the largest number, whose leading piece is infinite, and whose field is
    saturated, so that it adds nothing to the weights' gradients: those of the batch without
    it."""
    W, (y0, w) = _weights(), _inputs()
    W[0][:, 3] = 1e-30   # 3.4e38 * 1e-30: layer 1 at 3.4e8
    keep = np.arange(len(y0)) != 5
    y0[5, 3] = 3.4e38
    got = _grads(cuda, "f32", W, y0, w, adjoint)
    want = _grads(cuda, "f32", W, y0[keep], w[keep], adjoint)
    assert bool(torch.isfinite(got[0]).all())
    got[0] = got[0][torch.tensor(keep)]
    _close(got, want)


def test_large_weight(cuda):
    """A weight whose leading piece is infinite, on an activation that is zero."""
    W, (y0, w) = _weights(), _inputs()
    w *= np.float32(2.0 ** -10)   # keeps its delta finite
    W[0][7], W[1][7] = 0.0, -200.0
    W[2][:, 7] = 0.0
    want = _grads(cuda, "f32", W, y0, w)
    W[2][0, 7] = 3.4e38
    _close(_grads(cuda, "f32", W, y0, w), want)


def test_large_bias(cuda):
    """An activation whose leading piece is infinite, on weights that are zero: only its own
    column of W3's gradient is large."""
    W, (y0, w) = _weights(), _inputs()
    w *= np.float32(2.0 ** -10)
    W[4][:, 9] = 0.0
    want = _grads(cuda, "f32", W, y0, w)
    W[3][9] = 3.4e38
    got = _grads(cuda, "f32", W, y0, w)
    got[5][:, 9] = want[5][:, 9] = 0.0
    _close(got, want)


def test_one_small_trajectory(cuda):
    """Cotangents near the least number in one trajectory of a tile: its own gradient keeps its
    accuracy beside the others."""
    W, (y0, w) = _weights(), _inputs()
    want = _grads(cuda, "f32", W, y0, w)[0][5]
    s = 2.0 ** -116
    w[5] *= np.float32(s)
    got = _grads(cuda, "f32", W, y0, w)[0][5] / s
    assert float((got - want).abs().max() / want.abs().max()) < TOL


def test_small_inside(cuda):
    """Units whose slopes are near 2^-21 in both hidden layers: deltas near the least number from
    cotangents that are not."""
    W, (y0, w) = _weights(), _inputs()
    W[1][:] = W[3][:] = -15.0
    s = np.float32(2.0 ** -70)
    got = _grads(cuda, "f32", W, y0, w * s)
    _close([g / float(s) for g in got], _grads(cuda, "f32", W, y0, w))
